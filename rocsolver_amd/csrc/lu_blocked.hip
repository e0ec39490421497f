// lu_blocked.hip -- right-looking blocked LU and blocked triangular solves for
// any m, n (the path for matrices beyond the register-resident kernels).
//
// getrf, per block column of OUTER_NB columns (reference structure:
// library/src/lapack/roclapack_getrf.hpp:608-752, without rocBLAS):
//   1. panel_reg (lu_panel.hip): one workgroup per matrix factors 8 to 32
//      columns in registers with partial pivoting, applies its interchanges to
//      the rest of the block column and solves U12 = L11^-1 A12 there; the
//      block column's rows below are then updated (gemm_sub_kernel), panel
//      after panel or, for large batches of narrow panels, by halves;
//   2. outer_apply (lu_panel.hip): the block column's interchanges, composed
//      into one map, on all other columns, and U12 right of it;
//   3. gemm_sub_kernel: A22 -= L21 * U12 on MFMA (v_mfma_f64_16x16x4f64 /
//      v_mfma_f32_16x16x4f32), 64x64 tiles.
// Panels too tall for the registers: panel_kernel, interchanging rows inside
// the panel at each column in global memory, then every other column at once
// (roclapack_getf2.hpp:41-99 semantics: the same final rows), u12_kernel, one
// thread per column right of the panel, and the update.
// getrs (roclapack_getrs.hpp:117-150): the interchanges, then each triangle
// in 128-row tiles, one launch per tile (update by the tile before, then its
// own solve) or, with work for the whole chip, a launch for each.
#include "internal.hpp"
#include "mfma.hpp"
#include "quad_solve.hpp"
#include "rows_rule.hpp"

#include <climits>

namespace rsa
{

constexpr int PANEL_NB = 32; // width of the panel in global memory
constexpr int PANEL_THREADS = 512;
// A block column of this many bytes over the batch, in panels of at most 16
// columns, is factored by halves: updating every column right of each panel
// moves it through memory once per panel (448 column passes of 128 in panels
// of 16, 960 of 8), halves once per level (192, 256) at the price of a launch
// for U12 of the larger ones.  Measured: dgetrf 4096 x 128 x 64 1.40 -> 1.10
// ms, x 16 (64 MB) 0.69 -> 0.63, but x 4 0.52 -> 0.54; sgetrf 4096 x 128 x 64
// 0.55 -> 0.51, x 16 0.34 -> 0.36.  The batch decides the order of the work
// only: both group the sums by panel, so that a matrix's factors are the same
// bits in any batch.
constexpr int64_t BISECT_BYTES = int64_t(64) << 20;
constexpr int64_t MAX_GRID_YZ = 65535; // grid y/z limit: larger batches are launched in chunks

// ------------------------------------------------------------------ info
__global__ void reset_info_kernel(int* info, int bc)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if(i < bc)
        info[i] = 0;
}

rocblas_status reset_info(hipStream_t stream, int* info, int bc)
{
    if(bc <= 0)
        return rocblas_status_success;
    hipLaunchKernelGGL(reset_info_kernel, dim3(ceil_div(bc, 256)), dim3(256), 0, stream, info, bc);
    RSA_LAUNCH_CHECK();
    return rocblas_status_success;
}

// ------------------------------------------------------------ panel + trsm
template <typename T, bool PIVOT>
__global__ __launch_bounds__(PANEL_THREADS) void panel_kernel(int m, int n, Batch<T> AA, int lda,
                                                              int* __restrict__ ipivA,
                                                              int64_t strideP,
                                                              int* __restrict__ info, int j0,
                                                              int jb)
{
    constexpr int NT = PANEL_THREADS;
    constexpr int NW = NT / 64;
    __shared__ T s_key[NW];
    __shared__ int s_idx[NW];
    __shared__ T s_val[NW]; // each wavefront's candidate value
    __shared__ int s_swap[PANEL_NB]; // row interchanged with row j0 + k (itself: none)
    __shared__ int s_pos[2 * PANEL_NB]; // rows touched by the panel's interchanges
    __shared__ int s_src[2 * PANEL_NB]; // original row whose entries end at s_pos[q]
    __shared__ int s_cnt;

    const int64_t b = blockIdx.x;
    T* A = AA[b];
    const int tid = threadIdx.x;
    const int wid = tid / 64;
    const int lane = tid % 64;
    auto at = [&](int i, int j) -> T& { return A[i + int64_t(j) * lda]; };

    for(int k = 0; k < jb; ++k)
    {
        const int c = j0 + k;
        int p = c;
        T pv;
        if(PIVOT)
        {
            T key = T(-1), val = T(0);
            int idx = INT_MAX;
#pragma unroll 4
            for(int i = c + tid; i < m; i += NT)
            {
                const T a = at(i, c);
                T kk = pivot_key(a, i == c);
                if(kk > key)
                {
                    key = kk;
                    idx = i;
                    val = a;
                }
            }
            const int my_idx = idx;
            wave_argmax(key, idx);
            if(lane == 0)
            {
                s_key[wid] = key;
                s_idx[wid] = idx;
            }
            // the lane holding the winning row publishes its value (rows are
            // distinct across lanes), so no global read of it follows
            if(my_idx == idx && idx != INT_MAX)
                s_val[wid] = val;
            __syncthreads();
            // every thread combines the wavefronts' candidates itself (no
            // serial section and no second barrier)
            T bk = s_key[0];
            int bw = 0;
            p = s_idx[0];
            for(int w = 1; w < NW; ++w)
                if(s_key[w] > bk || (s_key[w] == bk && s_idx[w] < p))
                {
                    bk = s_key[w];
                    p = s_idx[w];
                    bw = w;
                }
            pv = s_val[bw];
            if(tid == 0)
            {
                ipivA[b * strideP + c] = p + 1;
                if(pv == T(0) && info[b] == 0)
                    info[b] = c + 1;
            }
        }
        else
        {
            pv = at(c, c);
            if(tid == 0 && pv == T(0) && info[b] == 0)
                info[b] = c + 1;
        }
        const bool nz = pv != T(0);
        if(tid == 0)
            s_swap[k] = (nz && p != c) ? p : c;
        // interchange rows c and p inside the panel (the other columns take
        // all of the panel's interchanges at once after it)
        const int jend = j0 + jb;
        if(nz && p != c)
        {
            for(int j = j0 + tid; j < jend; j += NT)
            {
                T t = at(c, j);
                at(c, j) = at(p, j);
                at(p, j) = t;
            }
        }
        __syncthreads();
        // scale the column and update the rest of the panel.  A zero pivot
        // leaves the column alone with pivoting (every candidate is zero) and
        // multiplies it by zero without (the reference npvt kernels keep the
        // scale at 0: roclapack_getf2_specialized_kernels.hpp:185-188,427-430)
        const T rcp = nz ? T(1) / pv : T(0);
        // the pivot row's panel entries right of c, then per row all loads
        // before any store, so they are in flight together
        T u[PANEL_NB];
#pragma unroll
        for(int q = 0; q < PANEL_NB; ++q)
        {
            const int j = j0 + q;
            u[q] = (j > c && j < jend) ? at(c, j) : T(0);
        }
        // two rows per pass (i and i + NT): both rows' loads are
        // issued before either row's stores
        for(int i = c + 1 + tid; i < m; i += 2 * NT)
        {
            const int i1 = i + NT;
            const bool has1 = i1 < m;
            T l0 = at(i, c);
            T l1 = has1 ? at(i1, c) : T(0);
            T v0[PANEL_NB], v1[PANEL_NB];
#pragma unroll
            for(int q = 0; q < PANEL_NB; ++q)
            {
                const int j = j0 + q;
                const bool in = j > c && j < jend;
                v0[q] = in ? at(i, j) : T(0);
                v1[q] = (in && has1) ? at(i1, j) : T(0);
            }
            if(nz || !PIVOT)
            {
                l0 *= rcp;
                l1 *= rcp;
                at(i, c) = l0;
                if(has1)
                    at(i1, c) = l1;
            }
#pragma unroll
            for(int q = 0; q < PANEL_NB; ++q)
            {
                const int j = j0 + q;
                if(j > c && j < jend)
                {
                    at(i, j) = fma_t(-l0, u[q], v0[q]);
                    if(has1)
                        at(i1, j) = fma_t(-l1, u[q], v1[q]);
                }
            }
        }
        __syncthreads();
    }

    // the panel's interchanges on every column outside it: composed into one
    // map of at most 2 jb rows (s_src[q]: the original row whose entries end
    // in row s_pos[q]), then each column reads those rows and writes them
    // back permuted
    if(PIVOT && n > jb)
    {
        if(wid == 0)
        {
            // lane q keeps slot q (row pos, source src); ballots find a row's
            // slot, a new row takes the next free one
            int pos = -1, src = -1, cnt = 0;
            for(int k = 0; k < jb; ++k)
            {
                const int r = j0 + k, r2 = s_swap[k];
                if(r2 == r) // uniform
                    continue;
                int qs[2];
#pragma unroll
                for(int h = 0; h < 2; ++h)
                {
                    const int row = h ? r2 : r;
                    const uint64_t hit = __builtin_amdgcn_ballot_w64(pos == row);
                    int q = hit ? __builtin_ffsll(hit) - 1 : cnt;
                    if(!hit)
                    {
                        if(lane == q)
                        {
                            pos = row;
                            src = row;
                        }
                        ++cnt;
                    }
                    qs[h] = q;
                }
                const int sa = __builtin_amdgcn_readlane(src, qs[0]);
                const int sb = __builtin_amdgcn_readlane(src, qs[1]);
                if(lane == qs[0])
                    src = sb;
                if(lane == qs[1])
                    src = sa;
            }
            if(lane < cnt)
            {
                s_pos[lane] = pos;
                s_src[lane] = src;
            }
            if(lane == 0)
                s_cnt = cnt;
        }
        __syncthreads();
        const int cnt = s_cnt;
        const int nout = n - jb; // columns left and right of the panel
        for(int e = tid; e < nout; e += NT)
        {
            const int j = e < j0 ? e : e + jb;
            T v[2 * PANEL_NB];
#pragma unroll
            for(int q = 0; q < 2 * PANEL_NB; ++q)
                v[q] = q < cnt ? at(s_src[q], j) : T(0);
#pragma unroll
            for(int q = 0; q < 2 * PANEL_NB; ++q)
                if(q < cnt)
                    at(s_pos[q], j) = v[q];
        }
        __syncthreads();
    }
}

// U12 = L11^-1 A12 for the columns right of a finished panel (L11 = the unit
// lower triangle of A[j0:j0+jb, j0:j0+jb]): one thread per column, 64
// columns per workgroup, L11 staged in LDS (zero outside jb x jb).
template <typename T>
__global__ __launch_bounds__(64) void u12_kernel(int n, Batch<T> AA, int lda, int j0, int jb,
                                                 int64_t boff)
{
    __shared__ T sL[PANEL_NB * PANEL_NB];
    const int64_t b = blockIdx.y + boff;
    T* A = AA[b];
    const int tid = threadIdx.x;
    for(int e = tid; e < PANEL_NB * PANEL_NB; e += 64)
    {
        const int i = e % PANEL_NB, k = e / PANEL_NB;
        sL[e] = (i < jb && k < jb) ? A[j0 + i + int64_t(j0 + k) * lda] : T(0);
    }
    __syncthreads();
    const int j = j0 + jb + blockIdx.x * 64 + tid;
    if(j >= n)
        return;
    T* col = A + int64_t(j) * lda + j0;
    T x[PANEL_NB];
#pragma unroll
    for(int i = 0; i < PANEL_NB; ++i)
        x[i] = i < jb ? col[i] : T(0);
    // L11 read through an offset that the optimiser must take as computed
    // from x[k] every two columns (an empty asm tied to x[k]), so its 496
    // entries are not all loaded ahead of the substitution (and spilled)
    const T* L = sL;
#pragma unroll
    for(int k = 0; k < PANEL_NB; ++k)
    {
        if((k & 1) == 0)
        {
            uint32_t lo = 0;
            asm volatile("" : "+v"(lo) : "v"(x[k]));
            L = sL + lo;
        }
#pragma unroll
        for(int i = k + 1; i < PANEL_NB; ++i)
            x[i] = fma_t(-L[i + k * PANEL_NB], x[k], x[i]);
    }
#pragma unroll
    for(int i = 0; i < PANEL_NB; ++i)
        if(i < jb)
            col[i] = x[i];
}

// ------------------------------------------------------------------ GEMM
// C[M x N] -= A[M x K] * B[K x N], column-major, one 64x64 tile per
// workgroup (4 waves, each 32x32 = 2x2 MFMA 16x16 blocks).  K goes through
// LDS in double-buffered chunks of 16, one barrier a chunk: the next chunk's
// global loads are in flight during this chunk's matrix instructions.  The
// operands are swapped (each 16x16 block is formed as its transpose: MFMA
// operand/result layouts in mfma.hpp), so 16 lanes read and write 16
// consecutive rows of C.
//
// Workgroups go round-robin to the 8 XCDs in launch order.  With 8 matrices
// or more a matrix's tiles are given to one XCD, so that its A and B panels
// are read into one L2.
constexpr int GT = 64; // tile
constexpr int GK = 16; // k chunk
constexpr int XCDS = 8;

// The products are summed and subtracted from C, in registers, GROUP values of
// k at a time: 32, so that the sums stay short (one sum over K = 128 made the
// errors of LU and solve 1.1 to 1.2 times larger on random matrices), or a
// panel's columns, so that one update by several panels rounds as an update by
// each of them does.  So C is read at the start, with A and B, which is also
// what an update inside a block column wants, a chain of two memory round trips
// rather than a stream (one n = 2000 system 10.6 -> 7.0 us a launch).
//
// TRANSA: the K x M transpose of A is stored; it goes through LDS by rows of
// the product, as B does by columns.
constexpr int GG = 32;

// Wavefronts a SIMD in groups of 32: n = 1024 x 64, FP32 with 4 in place of 5
// 2 % slower (three registers are spilled for 5), FP64 with 3 in place of 4 3 %.
// Shorter groups: the fewest registers win (6000 x 128 x 64 FP32, groups of 8,
// with 5 1.00 in place of 0.90 ms).
template <typename T, int GROUP, bool TRANSA>
constexpr int GEMM_WAVES = GROUP < 2 * GK ? 1 : sizeof(T) == 4 ? 5 : TRANSA ? 1 : 4;

template <typename T, int GROUP, bool TRANSA>
__global__ __launch_bounds__(256, (GEMM_WAVES<T, GROUP, TRANSA>)) void gemm_sub_kernel(
    int M, int N, int K, Batch<T> AA, int64_t offA, int lda, Batch<T> BB, int64_t offB, int ldb,
    Batch<T> CC, int64_t offC, int ldc, const int* __restrict__ skip, int bc, int tm,
    unsigned tile0, unsigned tiles)
{
    using M_ = mfma16<T>;
    using acc_t = typename M_::acc_t;
    // LDS strides that spread an MFMA operand read (16 rows or columns, 2
    // FP64 or 4 FP32 values of k per 32 or 64 lanes) over the banks
    constexpr int SR = GT + 16; // [k][i]
    constexpr int SC = GK + 1; // [j][k]
    constexpr int PT = GT * GK / 256; // entries of each operand per thread and chunk
    __shared__ T sA[2][TRANSA ? GT * SC : GK * SR];
    __shared__ T sB[2][GT * SC];

    const unsigned id = blockIdx.x;
    int64_t b;
    unsigned tile;
    if(bc >= XCDS)
    {
        b = int64_t(id / (XCDS * tiles)) * XCDS + id % XCDS;
        tile = tile0 + (id / XCDS) % tiles;
        if(b >= bc)
            return;
    }
    else
    {
        b = id / tiles;
        tile = tile0 + id % tiles;
    }
    if(skip && skip[b] != 0)
        return;
    const T* A = AA[b] + offA;
    const T* Bm = BB[b] + offB;
    T* C = CC[b] + offC;
    const int i0 = int(tile % tm) * GT;
    const int j0 = int(tile / tm) * GT;
    const int tid = threadIdx.x;
    const int wid = tid / 64;
    const int lane = tid % 64;
    const int wi = (wid % 2) * 32;
    const int wj = (wid / 2) * 32;

    acc_t acc[2][2];
#pragma unroll
    for(int s = 0; s < 2; ++s)
#pragma unroll
        for(int t = 0; t < 2; ++t)
            acc[s][t] = acc_t{0, 0, 0, 0};

    T c0[2][2][4];
    auto load_c = [&]() {
#pragma unroll
        for(int s = 0; s < 2; ++s)
#pragma unroll
            for(int t = 0; t < 2; ++t)
#pragma unroll
                for(int r = 0; r < 4; ++r)
                {
                    const int i = i0 + wi + s * 16 + lane % 16;
                    const int j = j0 + wj + t * 16 + M_::row(lane, r);
                    c0[s][t][r] = (i < M && j < N) ? C[i + int64_t(j) * ldc] : T(0);
                }
    };
    T ra[PT], rb[PT];
    auto load = [&](int k0) { // zero padded
#pragma unroll
        for(int t = 0; t < PT; ++t)
        {
            const int e = tid + 256 * t;
            const int i = i0 + (TRANSA ? e / GK : e % GT), k = k0 + (TRANSA ? e % GK : e / GT);
            ra[t] = (i < M && k < K) ? A[TRANSA ? k + int64_t(i) * lda : i + int64_t(k) * lda]
                                     : T(0);
            const int kb = k0 + e % GK, jb = j0 + e / GK;
            rb[t] = (kb < K && jb < N) ? Bm[kb + int64_t(jb) * ldb] : T(0);
        }
    };
    auto subtract = [&]() {
#pragma unroll
        for(int s = 0; s < 2; ++s)
#pragma unroll
            for(int t = 0; t < 2; ++t)
            {
#pragma unroll
                for(int r = 0; r < 4; ++r)
                    c0[s][t][r] -= acc[s][t][r];
                acc[s][t] = acc_t{0, 0, 0, 0};
            }
    };
    static_assert(GROUP % 4 == 0 && (GROUP == 2 * GK || GK % GROUP == 0), "whole groups");
    load(0);
    // The loop in place keeps C's addresses in registers for the stores, the
    // call does not: n = 1500 x 32 FP32 1 % faster so, groups of 8 (6000 x 128 x
    // 64 FP32) 4 % slower.
    if constexpr(GROUP == 2 * GK)
    {
#pragma unroll
        for(int s = 0; s < 2; ++s)
#pragma unroll
            for(int t = 0; t < 2; ++t)
#pragma unroll
                for(int r = 0; r < 4; ++r)
                {
                    const int i = i0 + wi + s * 16 + lane % 16;
                    const int j = j0 + wj + t * 16 + M_::row(lane, r);
                    c0[s][t][r] = (i < M && j < N) ? C[i + int64_t(j) * ldc] : T(0);
                }
    }
    else
        load_c();
    auto chunk = [&](int k0, int buf) {
#pragma unroll
        for(int t = 0; t < PT; ++t)
        {
            const int e = tid + 256 * t;
            sA[buf][TRANSA ? (e / GK) * SC + e % GK : (e / GT) * SR + e % GT] = ra[t];
            sB[buf][(e / GK) * SC + e % GK] = rb[t];
        }
        __syncthreads();
        if(k0 + GK < K) // uniform
            load(k0 + GK);
#pragma unroll
        for(int kk = 0; kk < GK; kk += 4)
        {
            T a[2], bv[2];
            const int k = kk + lane / 16;
#pragma unroll
            for(int s = 0; s < 2; ++s)
            {
                const int i = wi + s * 16 + lane % 16;
                a[s] = sA[buf][TRANSA ? i * SC + k : k * SR + i];
            }
#pragma unroll
            for(int t = 0; t < 2; ++t)
                bv[t] = sB[buf][(wj + t * 16 + lane % 16) * SC + k];
#pragma unroll
            for(int s = 0; s < 2; ++s)
#pragma unroll
                for(int t = 0; t < 2; ++t)
                    acc[s][t] = M_::run(bv[t], a[s], acc[s][t]);
            if(GROUP < 2 * GK && (k0 + kk + 4) % GROUP == 0)
            {
                subtract();
            }
        }
    };
    if constexpr(sizeof(T) == 8 && GROUP == 2 * GK)
    {
        // both chunks of a sum unrolled: its first products take a zero
        // constant (n = 1024 x 64 2 to 3 % faster; FP32 2 % slower)
        for(int k0 = 0; k0 < K; k0 += 2 * GK)
        {
            chunk(k0, 0);
            if(k0 + GK < K) // uniform
                chunk(k0 + GK, 1);
            subtract();
        }
    }
    else
    {
        int buf = 0;
        for(int k0 = 0; k0 < K; k0 += GK, buf ^= 1)
        {
            chunk(k0, buf);
            if(GROUP == 2 * GK && (buf == 1 || k0 + GK >= K)) // uniform
            {
                subtract();
            }
        }
    }

#pragma unroll
    for(int s = 0; s < 2; ++s)
    {
        const int i = i0 + wi + s * 16 + lane % 16;
#pragma unroll
        for(int t = 0; t < 2; ++t)
#pragma unroll
            for(int r = 0; r < 4; ++r)
            {
                const int j = j0 + wj + t * 16 + M_::row(lane, r);
                if(i < M && j < N)
                    C[i + int64_t(j) * ldc] = c0[s][t][r];
            }
    }
}

template <typename T>
static rocblas_status gemm_sub(hipStream_t stream, int M, int N, int K, Batch<T> A,
                               int64_t offA, int lda, Batch<T> B, int64_t offB, int ldb,
                               Batch<T> C, int64_t offC, int ldc, int bc, const int* skip,
                               int group = GG, bool transA = false)
{
    if(M <= 0 || N <= 0 || K <= 0 || bc <= 0)
        return rocblas_status_success;
    const int tm = ceil_div(M, GT);
    return launch_split(
        bc, int64_t(tm) * ceil_div(N, GT), 256, XCDS,
        [&](int64_t b0, int64_t nb, int64_t t0, int64_t nt) {
            const int64_t wgs = nt * (nb >= XCDS ? int64_t(ceil_div(nb, XCDS)) * XCDS : nb);
            const int* sk = skip ? skip + b0 : nullptr;
            auto go = [&](auto grp, auto tr) {
                hipLaunchKernelGGL(
                    (gemm_sub_kernel<T, decltype(grp)::value, decltype(tr)::value>),
                    dim3(unsigned(wgs)), dim3(256), 0, stream, M, N, K, batch_from(A, b0), offA,
                    lda, batch_from(B, b0), offB, ldb, batch_from(C, b0), offC, ldc, sk, int(nb),
                    tm, unsigned(t0), unsigned(nt));
            };
            using std::integral_constant;
            if(transA)
                go(integral_constant<int, GG>{}, std::true_type{});
            else if(group == 8)
                go(integral_constant<int, 8>{}, std::false_type{});
            else if(group == 16)
                go(integral_constant<int, 16>{}, std::false_type{});
            else
                go(integral_constant<int, GG>{}, std::false_type{});
            RSA_LAUNCH_CHECK();
            return rocblas_status_success;
        });
}

// ----------------------------------------------------------------- getrf
template <typename T>
rocblas_status getrf_blocked(hipStream_t stream, int m, int n, Batch<T> A, int lda, int* ipiv,
                             int64_t strideP, int* info, int bc, bool pivot)
{
    rocblas_status st = reset_info(stream, info, bc);
    if(st != rocblas_status_success)
        return st;
    const int kmax = m < n ? m : n;
    // C[r0:m, r0:jend] -= A[r0:m, j:r0] A[j:r0, r0:jend]
    auto update = [&](int j, int r0, int jend, int group = GG) {
        return gemm_sub<T>(stream, m - r0, jend - r0, r0 - j, A, r0 + int64_t(j) * lda, lda,
                           A, j + int64_t(r0) * lda, lda, A, r0 + int64_t(r0) * lda, lda, bc,
                           nullptr, group);
    };
    // Columns [j, j + w) of the block column [o0, oend) by halves: the left
    // half is factored, applied to the right half at once, then the right
    // half.  uend: U12 of a single panel is solved up to there.  The left half
    // is whole panels of one width and is applied with the roundings of panel
    // after panel, so that a matrix's factors do not depend on its batch.
    auto bisect = [&](auto&& self, int j, int w, int uend, int o0, int oend) -> rocblas_status {
        const int w0 = panel_reg_width<T>(m - j, lda);
        if(w <= w0)
            return panel_reg<T>(stream, m, A, lda, ipiv, strideP, info, j, w, o0, oend, uend, bc,
                                pivot);
        int w1 = w0;
        while(2 * w1 < w)
            w1 *= 2;
        for(int c = w0; c < w1; c += w0) // up to where fewer rows allow wider panels
            if(panel_reg_width<T>(m - j - c, lda) > w0)
                w1 = c;
        rocblas_status s = self(self, j, w1, w1 == w0 ? j + w : j + w1, o0, oend);
        if(s == rocblas_status_success && w1 > w0) // the panels have moved the rows already
            s = outer_apply<T>(stream, j + w, A, lda, ipiv, strideP, j, w1, bc, false, w0);
        if(s == rocblas_status_success)
            s = update(j, j + w1, j + w, w0);
        return s == rocblas_status_success ? self(self, j + w1, w - w1, j + w, o0, oend) : s;
    };
    for(int o0 = 0, nb = 0; o0 < kmax; o0 += nb)
    {
        if(panel_reg_width<T>(m - o0, lda))
        {
            // a block column of OUTER_NB columns: its panels in registers,
            // each applied to the rest of the block only, then the block to
            // the rest of the matrix, so the trailing matrix is read and
            // written once per OUTER_NB columns
            nb = (kmax - o0) < OUTER_NB ? (kmax - o0) : OUTER_NB;
            const int oend = o0 + nb;
            const int w0 = panel_reg_width<T>(m - o0, lda);
            if(w0 <= 16 && int64_t(bc) * (m - o0) * nb * int64_t(sizeof(T)) >= BISECT_BYTES)
                st = bisect(bisect, o0, nb, oend, o0, oend);
            else
                for(int j = o0, jb = 0; j < oend && st == rocblas_status_success; j += jb)
                {
                    const int w = panel_reg_width<T>(m - j, lda);
                    jb = (oend - j) < w ? (oend - j) : w;
                    st = panel_reg<T>(stream, m, A, lda, ipiv, strideP, info, j, jb, o0, oend,
                                      oend, bc, pivot);
                    if(st == rocblas_status_success)
                        st = update(j, j + jb, oend);
                }
            if(st != rocblas_status_success)
                return st;
            st = outer_apply<T>(stream, n, A, lda, ipiv, strideP, o0, nb, bc, pivot);
            if(st == rocblas_status_success)
                st = update(o0, oend, n);
            if(st != rocblas_status_success)
                return st;
            continue;
        }
        // panels too tall for the registers, factored in global memory
        nb = (kmax - o0) < PANEL_NB ? (kmax - o0) : PANEL_NB;
        const int r0 = o0 + nb;
        if(pivot)
            hipLaunchKernelGGL((panel_kernel<T, true>), dim3(bc), dim3(PANEL_THREADS), 0, stream, m,
                               n, A, lda, ipiv, strideP, info, o0, nb);
        else
            hipLaunchKernelGGL((panel_kernel<T, false>), dim3(bc), dim3(PANEL_THREADS), 0, stream,
                               m, n, A, lda, ipiv, strideP, info, o0, nb);
        RSA_LAUNCH_CHECK();
        if(r0 < n)
            for(int64_t b0 = 0; b0 < bc; b0 += MAX_GRID_YZ)
            {
                const int cnt = int((bc - b0) < MAX_GRID_YZ ? (bc - b0) : MAX_GRID_YZ);
                hipLaunchKernelGGL((u12_kernel<T>), dim3(ceil_div(n - r0, 64), cnt), dim3(64), 0,
                                   stream, n, A, lda, o0, nb, b0);
                RSA_LAUNCH_CHECK();
            }
        st = update(o0, r0, n);
        if(st != rocblas_status_success)
            return st;
    }
    return rocblas_status_success;
}

// ----------------------------------------------------------------- laswp
// One thread per column; the interchanges of one column run in order
// (rocauxiliary_laswp.hpp:41-62).
template <typename T>
__global__ __launch_bounds__(256) void laswp_kernel(int ncols, Batch<T> AA, int lda, int k1,
                                                    int k2, const int* __restrict__ ipivA,
                                                    int64_t strideP, int incx,
                                                    const int* __restrict__ skip, int64_t boff)
{
    const int64_t b = blockIdx.y + boff;
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if(c >= ncols || (skip && skip[b] != 0))
        return;
    T* A = AA[b] + int64_t(c) * lda;
    const int* ipiv = ipivA + b * strideP;
    int start, end, inc;
    if(incx < 0)
    {
        start = k2;
        end = k1 - 1;
        inc = -1;
        incx = -incx;
    }
    else
    {
        start = k1;
        end = k2 + 1;
        inc = 1;
    }
    for(int i = start; i != end; i += inc)
    {
        const int ex = ipiv[k1 + (i - k1) * incx - 1];
        // a pivot outside the column's storage is ignored instead of addressed
        if(ex != i && ex >= 1 && ex <= lda)
        {
            T t = A[i - 1];
            A[i - 1] = A[ex - 1];
            A[ex - 1] = t;
        }
    }
}

template <typename T>
rocblas_status laswp(hipStream_t stream, int ncols, Batch<T> A, int lda, int k1, int k2,
                     const int* ipiv, int64_t strideP, int incx, int bc, const int* skip_info)
{
    if(ncols <= 0 || bc <= 0)
        return rocblas_status_success;
    for(int64_t b0 = 0; b0 < bc; b0 += MAX_GRID_YZ)
    {
        const int nb = int((bc - b0) < MAX_GRID_YZ ? (bc - b0) : MAX_GRID_YZ);
        dim3 grid(ceil_div(ncols, 256), nb);
        hipLaunchKernelGGL((laswp_kernel<T>), grid, dim3(256), 0, stream, ncols, A, lda, k1, k2,
                           ipiv, strideP, incx, skip_info, b0);
        RSA_LAUNCH_CHECK();
    }
    return rocblas_status_success;
}

// --------------------------------------------------------------- row order
// B <- P B (or with inverse, P^T B) for the interchanges of ipiv (1-based,
// LAPACK order; a pivot outside [1, n] is ignored), n <= 1024 R rows.
//
// The interchanges are composed in blocks of 64: a wavefront follows the 64
// rows of a block and the 64 rows they are interchanged with through the
// block's steps, and one wavefront then applies the blocks' maps in order to
// a table of the rows in LDS.  Every column is gathered through the table.
// (Following every row through all n interchanges took 161 us at n = 2000,
// and laswp_kernel, two dependent global accesses per row, 154 us; this
// kernel takes 17 us there.)
constexpr int PERM_THREADS = 1024;
constexpr int PERM_COLS = 8; // columns per workgroup

template <typename T, int R>
__global__ __launch_bounds__(PERM_THREADS) void permute_rows_kernel(
    int n, int nrhs, Batch<T> BB, int ldb, const int* __restrict__ ipivA, int64_t strideP,
    int inverse, const int* __restrict__ skip, unsigned group0, int64_t boff)
{
    constexpr int ROWS = PERM_THREADS * R;
    __shared__ unsigned short s_row[ROWS]; // row now at each position
    __shared__ unsigned short s_pos[ROWS]; // block maps: the rows interchanged with,
    __shared__ unsigned short s_src[2][ROWS]; // and where both kinds come from
    const int64_t b = blockIdx.y + boff;
    if(skip && skip[b] != 0)
        return;
    T* Bm = BB[b];
    const int* ipiv = ipivA + b * strideP;
    const int tid = threadIdx.x;
    const int lane = tid % 64;
    const int nblk = (n + 63) / 64;
    for(int i = tid; i < ROWS; i += PERM_THREADS)
        s_row[i] = (unsigned short)i;
    for(int blk = tid / 64; blk < nblk; blk += PERM_THREADS / 64) // one wavefront per block
    {
        const int base = 64 * blk, i = base + lane;
        int p = i < n ? ipiv[i] - 1 : i;
        p = (p >= 0 && p < n) ? p : i;
        int s0 = i, s1 = p;
#pragma unroll 8
        for(int e = 0; e < 64; ++e)
        {
            // back through the block's steps, the last one applied first
            const int k = inverse ? e : 63 - e;
            const int row = base + k;
            const int q = __builtin_amdgcn_readlane(p, k);
            s0 = s0 == row ? q : (s0 == q ? row : s0);
            s1 = s1 == row ? q : (s1 == q ? row : s1);
        }
        s_src[0][i] = (unsigned short)s0;
        // a partner inside the block is one of its rows; one met twice is
        // moved twice, the same row to the same place
        const bool inside = p >= base && p < base + 64;
        s_pos[i] = (unsigned short)(inside ? i : p);
        s_src[1][i] = (unsigned short)(inside ? s0 : s1);
    }
    __syncthreads();
    if(tid < 64)
        for(int e = 0; e < nblk; ++e)
        {
            const int i = 64 * (inverse ? nblk - 1 - e : e) + lane;
            const int pos = s_pos[i];
            const unsigned short r0 = s_row[s_src[0][i]], r1 = s_row[s_src[1][i]];
            wave_sync();
            s_row[i] = r0;
            s_row[pos] = r1;
            wave_sync();
        }
    __syncthreads();
    int src[R];
#pragma unroll
    for(int r = 0; r < R; ++r)
        src[r] = s_row[tid + r * PERM_THREADS];
    const int c0 = int(group0 + blockIdx.x) * PERM_COLS;
    constexpr int UC = R <= 4 ? 4 : 2; // columns in flight
    for(int c1 = 0; c1 < PERM_COLS && c0 + c1 < nrhs; c1 += UC) // uniform
    {
        T x[UC][R];
#pragma unroll
        for(int u = 0; u < UC; ++u)
#pragma unroll
            for(int r = 0; r < R; ++r)
                x[u][r] = (tid + r * PERM_THREADS < n && c0 + c1 + u < nrhs)
                              ? Bm[src[r] + int64_t(c0 + c1 + u) * ldb]
                              : T(0);
        __syncthreads(); // the loads of these columns are done
#pragma unroll
        for(int u = 0; u < UC; ++u)
#pragma unroll
            for(int r = 0; r < R; ++r)
                if(tid + r * PERM_THREADS < n && c0 + c1 + u < nrhs)
                    Bm[tid + r * PERM_THREADS + int64_t(c0 + c1 + u) * ldb] = x[u][r];
    }
}

template <typename T>
static rocblas_status permute_rows(hipStream_t stream, int n, int nrhs, Batch<T> B, int ldb,
                                   const int* ipiv, int64_t strideP, bool inverse, int bc,
                                   const int* skip)
{
    if(n > 8 * PERM_THREADS)
        return laswp<T>(stream, nrhs, B, ldb, 1, n, ipiv, strideP, inverse ? -1 : 1, bc, skip);
    for(int64_t b0 = 0; b0 < bc; b0 += MAX_GRID_YZ)
    {
        const int nb = int((bc - b0) < MAX_GRID_YZ ? (bc - b0) : MAX_GRID_YZ);
        auto go = [&](auto r) {
            return launch_split(
                1, ceil_div(nrhs, PERM_COLS), PERM_THREADS, 1,
                [&](int64_t, int64_t, int64_t g0, int64_t ng) {
                    hipLaunchKernelGGL((permute_rows_kernel<T, decltype(r)::value>),
                                       dim3(unsigned(ng), nb), dim3(PERM_THREADS), 0, stream, n,
                                       nrhs, B, ldb, ipiv, strideP, int(inverse), skip,
                                       unsigned(g0), b0);
                    RSA_LAUNCH_CHECK();
                    return rocblas_status_success;
                });
        };
        const rocblas_status st = n <= PERM_THREADS       ? go(std::integral_constant<int, 1>{})
                                  : n <= 2 * PERM_THREADS ? go(std::integral_constant<int, 2>{})
                                  : n <= 4 * PERM_THREADS ? go(std::integral_constant<int, 4>{})
                                                          : go(std::integral_constant<int, 8>{});
        if(st != rocblas_status_success)
            return st;
    }
    return rocblas_status_success;
}

// ------------------------------------------------------------ substitution
// One step of a blocked triangular solve of op(A) X = B in place: every
// 128-row tile of the grid subtracts its block of op(A) times the solved tile
// `prev` (-1: none), and the workgroups of tile `next` then solve their
// diagonal block, so a step is one launch and the next step's solve does not
// wait for a launch of its own.
// KIND: 0 = L unit lower (forward), 1 = U non-unit upper (backward), 2 = U^T
// (forward, non-unit), 3 = L^T (backward, unit).
//
// COLS right-hand sides per workgroup (8 wavefronts: COLS / 16 groups of
// columns times the rest as groups of rows).  The products run on the matrix
// cores straight from memory (operands swapped, so that 16 lanes hold 16
// consecutive rows), with half of a wavefront's loads or all of them in
// flight.  The workgroup that solves holds its triangle of op(A) in LDS,
// loaded before the update: 32-row diagonal blocks are solved by four lanes
// per column, the rest of the tile updated by matrix-core products; a
// wavefront owns 16 columns there.
//
// Bound by latency: n / 128 dependent steps per triangle.  A thread per
// column solving 64-row blocks, with the update in a launch of its own, took
// 1.7 ms for both triangles at n = 1024 x 64, 8 right-hand sides (transposed)
// and 3.1 ms for one system of n = 2000; this kernel takes 0.69 and 0.80 ms.
// Where there is work for the whole chip (trsm_many) a step only solves, and
// gemm_sub_kernel updates: the same sums, the same bits.
constexpr int ST = 128; // tile rows
constexpr int SD = 32; // diagonal block rows
constexpr int STEP_THREADS = 512;

template <typename T, int KIND, int COLS>
__global__ __launch_bounds__(STEP_THREADS) void trsm_step_kernel(int n, int nrhs, Batch<T> AA,
                                                                 int lda, Batch<T> BB, int ldb,
                                                                 const int* __restrict__ skip,
                                                                 int prev, int next, int tile0,
                                                                 unsigned group0, int64_t boff)
{
    using M = mfma16<T>;
    constexpr bool LOWER = KIND == 0 || KIND == 2;
    constexpr bool UNIT = KIND == 0 || KIND == 3;
    constexpr bool TRANS = KIND >= 2;
    constexpr int CG = COLS / 16, RG = STEP_THREADS / 64 / CG; // groups of columns, of rows
    constexpr int RT = ST / 16 / RG; // 16-row tiles per wavefront
    constexpr int LS = ST + 1;
    constexpr int ND = ST / SD;
    __shared__ T sB[COLS * LS];
    // 32x32 blocks (i, k) of the triangle at i (i + 1) / 2 + k (i >= k, by
    // the block's row and column, exchanged for an upper triangle)
    __shared__ __align__(16) T sD[ND * (ND + 1) / 2][SD * SD];

    const int64_t b = blockIdx.z + boff;
    if(skip && skip[b] != 0)
        return;
    const T* A = AA[b];
    T* Bm = BB[b];
    const int tid = threadIdx.x;
    const int wid = tid / 64;
    const int lane = tid % 64;
    const int tile = tile0 + blockIdx.y;
    const int r0 = tile * ST;
    const int c0 = int(group0 + blockIdx.x) * COLS + 16 * (wid % CG); // this wavefront's columns
    const int wr = 16 * RT * (wid / CG); // and rows of the tile, in the update
    const bool solve = tile == next; // uniform
    auto op = [&](int i, int k) -> T {
        return TRANS ? A[k + int64_t(i) * lda] : A[i + int64_t(k) * lda];
    };
    auto block = [](int i, int k) { return i > k ? i * (i + 1) / 2 + k : k * (k + 1) / 2 + i; };

    if(solve) // the triangle of op(A), columns of each block contiguous; past n: the identity
    {
#pragma unroll
        for(int bi = 0; bi < ND; ++bi)
#pragma unroll
            for(int bk = 0; bk < ND; ++bk)
                if(LOWER ? bi >= bk : bi <= bk)
#pragma unroll
                    for(int h = 0; h < SD * SD / STEP_THREADS; ++h)
                    {
                        // memory order along the column of A
                        const int e = tid + h * STEP_THREADS, x = e % SD, y = e / SD;
                        const int i = TRANS ? y : x, k = TRANS ? x : y;
                        const int gi = r0 + SD * bi + i, gk = r0 + SD * bk + k;
                        sD[block(bi, bk)][k * SD + i]
                            = (gi < n && gk < n) ? op(gi, gk) : (gi == gk ? T(1) : T(0));
                    }
    }

    // this wavefront's right-hand sides: register r of tile t holds row wr + 16 t
    // + lane % 16, column M::row(lane, r)
    T x[RT][4];
#pragma unroll
    for(int t = 0; t < RT; ++t)
#pragma unroll
        for(int r = 0; r < 4; ++r)
        {
            const int i = r0 + wr + 16 * t + (lane & 15), c = c0 + M::row(lane, r);
            x[t][r] = i < n && c < nrhs ? Bm[i + int64_t(c) * ldb] : T(0);
        }
    const int col = c0 + (lane & 15);
    if(prev >= 0)
    {
        typename M::acc_t acc[RT];
#pragma unroll
        for(int t = 0; t < RT; ++t)
            acc[t] = typename M::acc_t{0, 0, 0, 0};
        const int k0 = prev * ST;
        constexpr int KS = RT == 1 ? 16 : 8; // matrix-core steps whose loads are in flight
#pragma unroll 1
        for(int kk = 0; kk < ST; kk += 4 * KS)
        {
            T bv[KS], av[KS][RT];
#pragma unroll
            for(int q = 0; q < KS; ++q)
            {
                const int k = k0 + kk + 4 * q + (lane >> 4);
                bv[q] = (k < n && col < nrhs) ? Bm[k + int64_t(col) * ldb] : T(0);
#pragma unroll
                for(int t = 0; t < RT; ++t)
                {
                    const int i = r0 + wr + 16 * t + (lane & 15);
                    av[q][t] = (i < n && k < n) ? op(i, k) : T(0);
                }
            }
#pragma unroll
            for(int q = 0; q < KS; ++q)
#pragma unroll
                for(int t = 0; t < RT; ++t)
                {
                    acc[t] = M::run(bv[q], av[q][t], acc[t]);
                    if((4 * q + 4) % GG == 0) // sums of GG products, as gemm_sub_kernel's
                    {
#pragma unroll
                        for(int r = 0; r < 4; ++r)
                            x[t][r] -= acc[t][r];
                        acc[t] = typename M::acc_t{0, 0, 0, 0};
                    }
                }
        }
    }
#pragma unroll
    for(int t = 0; t < RT; ++t)
    {
        const int li = wr + 16 * t + (lane & 15);
        const int i = r0 + li;
#pragma unroll
        for(int r = 0; r < 4; ++r)
        {
            const int c = c0 + M::row(lane, r);
            if(solve)
                sB[(16 * (wid % CG) + M::row(lane, r)) * LS + li] = x[t][r];
            else if(i < n && c < nrhs)
                Bm[i + int64_t(c) * ldb] = x[t][r];
        }
    }
    if(!solve)
        return;
    __syncthreads();
    if(wid >= CG || c0 >= nrhs) // one wavefront per 16 columns from here on
        return;
    T* colB = sB + 16 * wid * LS;
#pragma unroll
    for(int step = 0; step < ND; ++step)
    {
        const int d = LOWER ? step : ND - 1 - step;
        if(r0 + SD * d < n) // uniform
        {
            {
                T x[SD / 4];
                T* xp = colB + (lane >> 2) * LS + SD * d + (lane & 3);
#pragma unroll
                for(int t = 0; t < SD / 4; ++t)
                    x[t] = xp[4 * t];
                quad_solve<T, SD, LOWER, UNIT>(sD[block(d, d)], lane, x);
#pragma unroll
                for(int t = 0; t < SD / 4; ++t)
                    xp[4 * t] = x[t];
            }
            wave_sync();
            T bv[SD / 4];
#pragma unroll
            for(int ks = 0; ks < SD / 4; ++ks)
                bv[ks] = colB[(lane & 15) * LS + SD * d + 4 * ks + (lane >> 4)];
#pragma unroll
            for(int t = 0; t < ST / 16; ++t)
            {
                const int e = t / 2; // the 32-row block of these 16 rows
                if(LOWER ? e > d : e < d)
                {
                    typename M::acc_t u = {0, 0, 0, 0};
#pragma unroll
                    for(int ks = 0; ks < SD / 4; ++ks)
                        u = M::run(sD[block(e, d)][(4 * ks + (lane >> 4)) * SD + 16 * (t & 1)
                                                   + (lane & 15)],
                                   bv[ks], u);
#pragma unroll
                    for(int r = 0; r < 4; ++r)
                        colB[(lane & 15) * LS + 16 * t + M::row(lane, r)] -= u[r];
                }
            }
            wave_sync();
        }
    }
    for(int c = 0; c < 16; ++c)
        if(c0 + c < nrhs) // uniform
            for(int i = lane; i < ST && r0 + i < n; i += 64)
                Bm[r0 + i + int64_t(c0 + c) * ldb] = colB[c * LS + i];
}

// One triangle of A (KIND as above) against all right-hand sides.
template <typename T, int KIND>
static rocblas_status trsm_blocked(hipStream_t stream, int n, int nrhs, Batch<T> A, int lda,
                                   Batch<T> B, int ldb, int bc, const int* skip)
{
    constexpr bool LOWER = KIND == 0 || KIND == 2;
    constexpr bool TRANS = KIND >= 2;
    constexpr int WIDE = sizeof(T) == 8 ? 64 : 128; // what the LDS holds
    const int tiles = ceil_div(n, ST);
    const bool many = trsm_many<T>(TRANS, tiles, nrhs, bc);
    const int cols = nrhs <= 16 ? 16 : nrhs <= 32 || !many ? 32 : nrhs <= 64 ? 64 : WIDE;
    for(int s = 0; s < tiles; ++s)
    {
        // step s solves tile `next`, after the update by the tile before
        // unless the updates have launches of their own
        const int next = LOWER ? s : tiles - 1 - s;
        const int prev = s == 0 || many ? -1 : (LOWER ? s - 1 : next + 1);
        const int cnt = prev < 0 ? 1 : tiles - s; // tiles not solved yet
        const int tile0 = LOWER || prev < 0 ? next : 0;
        for(int64_t b0 = 0; b0 < bc; b0 += MAX_GRID_YZ)
        {
            const int nb = int((bc - b0) < MAX_GRID_YZ ? (bc - b0) : MAX_GRID_YZ);
            // right-hand sides in x: more than 65535 groups of them are allowed
            const rocblas_status st = launch_split(
                1, ceil_div(nrhs, cols), STEP_THREADS, 1,
                [&](int64_t, int64_t, int64_t g0, int64_t ng) {
                    auto go = [&](auto c) {
                        hipLaunchKernelGGL((trsm_step_kernel<T, KIND, decltype(c)::value>),
                                           dim3(unsigned(ng), cnt, nb), dim3(STEP_THREADS), 0,
                                           stream, n, nrhs, A, lda, B, ldb, skip, prev, next, tile0,
                                           unsigned(g0), b0);
                    };
                    if(cols == 16)
                        go(std::integral_constant<int, 16>{});
                    else if(cols == 32)
                        go(std::integral_constant<int, 32>{});
                    else if(cols == 64)
                        go(std::integral_constant<int, 64>{});
                    else
                        go(std::integral_constant<int, WIDE>{});
                    RSA_LAUNCH_CHECK();
                    return rocblas_status_success;
                });
            if(st != rocblas_status_success)
                return st;
        }
        if(many)
        {
            const int k0 = next * ST, k1 = k0 + ST < n ? k0 + ST : n;
            const int r0 = LOWER ? k1 : 0, r1 = LOWER ? n : k0; // the tiles not solved yet
            const int64_t offA = TRANS ? k0 + int64_t(r0) * lda : r0 + int64_t(k0) * lda;
            const rocblas_status st = gemm_sub<T>(stream, r1 - r0, nrhs, k1 - k0, A, offA, lda, B,
                                                  k0, ldb, B, r0, ldb, bc, skip, GG, TRANS);
            if(st != rocblas_status_success)
                return st;
        }
    }
    return rocblas_status_success;
}

template <typename T>
rocblas_status getrs_blocked(hipStream_t stream, bool trans, int n, int nrhs, Batch<T> A, int lda,
                             const int* ipiv, int64_t strideP, Batch<T> B, int ldb, int bc,
                             bool pivot, const int* skip)
{
    if(n <= 0 || nrhs <= 0 || bc <= 0)
        return rocblas_status_success;
    rocblas_status st = rocblas_status_success;
    if(!trans && pivot)
        st = permute_rows<T>(stream, n, nrhs, B, ldb, ipiv, strideP, false, bc, skip);
    if(st == rocblas_status_success)
        st = trans ? trsm_blocked<T, 2>(stream, n, nrhs, A, lda, B, ldb, bc, skip)
                   : trsm_blocked<T, 0>(stream, n, nrhs, A, lda, B, ldb, bc, skip);
    if(st == rocblas_status_success)
        st = trans ? trsm_blocked<T, 3>(stream, n, nrhs, A, lda, B, ldb, bc, skip)
                   : trsm_blocked<T, 1>(stream, n, nrhs, A, lda, B, ldb, bc, skip);
    if(st == rocblas_status_success && trans && pivot)
        st = permute_rows<T>(stream, n, nrhs, B, ldb, ipiv, strideP, true, bc, skip);
    return st;
}

#define RSA_INST(T)                                                                              \
    template rocblas_status getrf_blocked<T>(hipStream_t, int, int, Batch<T>, int, int*, int64_t, \
                                             int*, int, bool);                                   \
    template rocblas_status getrs_blocked<T>(hipStream_t, bool, int, int, Batch<T>, int,          \
                                             const int*, int64_t, Batch<T>, int, int, bool,       \
                                             const int*);                                        \
    template rocblas_status laswp<T>(hipStream_t, int, Batch<T>, int, int, int, const int*,       \
                                     int64_t, int, int, const int*);
RSA_INST(float)
RSA_INST(double)
#undef RSA_INST

} // namespace rsa
