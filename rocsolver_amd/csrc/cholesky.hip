// cholesky.hip -- batched Cholesky factorisation (potf2 / potrf), solve with
// the factor (potrs) and factor-and-solve (posv), uplo lower (A = L L^T) or
// upper (A = U^T U).  Only the referenced triangle is read or written.
//
// Factorisation: one workgroup per matrix, left-looking over 32-column block
// columns:
//   1. every row of the block column subtracts its products with the finished
//      columns on the matrix cores, 16 rows x 32 columns per step and
//      wavefront, operands straight from memory.  v_mfma_*_16x16x4 adds its
//      four products to the accumulator as a chain of fused multiply-adds
//      with k increasing (checked bit for bit on gfx950, FP32 and FP64,
//      denormals included), so accumulators that start at A and take -L as
//      one operand run the unblocked order of operations;
//   2. one wavefront factors the diagonal block in registers (right-looking;
//      column k reaches the other lanes through LDS);
//   3. the rows below solve against it, four lanes per row, multiplying by
//      the stored reciprocals, and the block column is written.
// Per entry the order of operations is that of the reference's unblocked
// potf2 (library/src/lapack/roclapack_potf2.hpp:160-250): t = a_jj minus the
// squares of row j's finished entries (one fma each, k increasing); t <= 0 ->
// info = first j + 1, a_jj = t and the column below is scaled by 0, and the
// factorisation goes on (sqrtDiagOnward, :10-37); otherwise a_jj = sqrt(t)
// and the entries below are (a_ij minus their products, k increasing) times
// 1 / a_jj.  So the factor equals the oracle's restatement bit for bit; the
// reference's own dot/gemv reductions differ from it by rounding only.
//
// Solve: for n <= 512 one workgroup per system with the tile solver of the LU
// path (tile_solve.hpp) or, for large batches of few right-hand sides, its row
// solver (trsv_rows.hpp, rows_rule.hpp), on non-unit triangles: L then L^T, or U^T then U
// (library/src/lapack/roclapack_potrs.hpp:121-148), with the same operations
// per row; larger orders use one thread per (system, right-hand side)
// substitution.
#include "mfma.hpp"
#include "quad_solve.hpp"
#include "rows_rule.hpp"
#include "tile_solve.hpp"
#include "trsv_rows.hpp"

#include <cmath>

namespace rsa
{

constexpr int CHB = 32; // block-column width
constexpr int CHR = 2; // 16-row groups per wavefront and pass

// Element (i, j), i >= j, of the lower factor L: A[i + j lda] with lower
// storage, A[j + i lda] with upper storage (which holds U = L^T).
template <typename T, bool UP>
struct LowerView
{
    T* a;
    int64_t lda;
    __device__ __forceinline__ T& operator()(int i, int j) const
    {
        return UP ? a[j + i * lda] : a[i + j * lda];
    }
    // distance between (i, j) and (i, j + 1)
    __device__ __forceinline__ int64_t next_col() const
    {
        return UP ? 1 : lda;
    }
};

// One row of the block column against the factored diagonal block, four lanes
// per row: lane s = lane & 3 holds entries 4 t + s in x[t].  x_k times the
// reciprocal 1 / l_kk, then x_m -= x_k l_mk for m > k.
template <typename T, int K = 0>
__device__ __forceinline__ void chol_row_solve(const T* L11, const T* res, int lane,
                                               T (&x)[CHB / 4])
{
    if constexpr(K < CHB)
    {
        if constexpr(K % 4 == 0)
        {
            const uint32_t zero = after(x);
            L11 += zero;
            res += zero;
        }
        const int s = lane & 3;
        const T y = x[K / 4] * res[K];
        x[K / 4] = s == K % 4 ? y : x[K / 4];
        const T xk = quad_broadcast<K % 4>(x[K / 4]);
        const T* col = L11 + K * CHB;
        if constexpr(K % 4 < 3)
        {
            const T z = fma_t(-xk, col[K / 4 * 4 + s], x[K / 4]);
            x[K / 4] = s > K % 4 ? z : x[K / 4];
        }
#pragma unroll
        for(int t = K / 4 + 1; t < CHB / 4; ++t)
            x[t] = fma_t(-xk, col[4 * t + s], x[t]);
        chol_row_solve<T, K + 1>(L11, res, lane, x);
    }
}

// Bound by latency: the chain of n pivots (square root, reciprocal and scaling
// of one column after the other on one wavefront), the row solves and the
// operand loads.  So small workgroups and 128 registers: four matrices share
// a CU, and the matrix-core products of one run under the pivots of another.
// n = 300 x 1024 FP64: 0.72 ms (three matrices per CU: 0.78); one thread per
// row with vector fused multiply-adds took 4.14 ms.  The 128 registers leave
// FP64 160 bytes a lane in scratch beyond n = 64.
template <typename T, int NT, bool UP>
__global__ __launch_bounds__(NT, NT == 64 ? 2 : 4) void potrf_kernel(int n, Batch<T> AA, int lda,
                                                      int* __restrict__ info)
{
    using M = mfma16<T>;
    constexpr int NW = NT / 64;
    constexpr int TS = CHB + 1; // row stride of the exchange buffers
    constexpr int KS = 2; // matrix-core steps whose loads are in flight
    __shared__ T sX[NW > 2 ? NW : 2][16 * TS]; // 16 rows per wavefront; first the diagonal block
    __shared__ T sL11[CHB * CHB]; // the factored diagonal block, by columns
    __shared__ T sres[CHB]; // 1 / l_jj, or 0 after a non-positive pivot
    __shared__ int sinfo;

    const int tid = threadIdx.x;
    const int wid = tid >> 6;
    const int64_t b = blockIdx.x;
    const LowerView<T, UP> L{AA[b], lda};
    if(tid == 0)
        sinfo = 0;
    for(int e = tid; e < CHB * CHB; e += NT)
        sL11[e] = T(0); // above the diagonal: read, never used

    for(int c0 = 0; c0 < n; c0 += CHB)
    {
        const int jb = n - c0 < CHB ? n - c0 : CHB;
        const int groups = (n - c0 + 15) / 16; // the first two hold the diagonal block
        for(int g0 = 0; g0 < groups; g0 += NW * CHR) // uniform
        {
            // group t of this wavefront and pass: rows c0 + 16 (g0 + wid + t NW) ...
            // lane & 15 is the row, register r the column M::row(lane, r).
            // Rows past n repeat row n - 1, entries above the diagonal the
            // diagonal's, and are not stored.  (In every phase the lane comes
            // from an opaque thread id: addresses and masks formed from it at
            // entry would stay live through all of them.)
            const int lane = fresh_tid() & 63;
            typename M::acc_t acc[CHR][2];
            const T* pa[CHR];
#pragma unroll
            for(int t = 0; t < CHR; ++t)
            {
                const int i = c0 + 16 * (g0 + wid + t * NW) + (lane & 15);
                const int row = i < n ? i : n - 1;
                pa[t] = &L(row, lane >> 4);
#pragma unroll
                for(int ct = 0; ct < 2; ++ct)
#pragma unroll
                    for(int r = 0; r < 4; ++r)
                    {
                        const int j = c0 + 16 * ct + M::row(lane, r);
                        acc[t][ct][r] = L(row, j < row ? j : row);
                    }
            }
            // ---- 1. products with the finished columns 0 .. c0-1
            const T* pb[2];
#pragma unroll
            for(int ct = 0; ct < 2; ++ct)
            {
                const int j = c0 + 16 * ct + (lane & 15);
                pb[ct] = &L(j < n ? j : n - 1, lane >> 4);
            }
            const int64_t step = 4 * L.next_col();
            T av[2][KS][CHR], bv[2][KS][2];
            auto load = [&](int h) {
#pragma unroll
                for(int q = 0; q < KS; ++q)
                {
#pragma unroll
                    for(int ct = 0; ct < 2; ++ct)
                    {
                        bv[h][q][ct] = *pb[ct];
                        pb[ct] += step;
                    }
#pragma unroll
                    for(int t = 0; t < CHR; ++t)
                    {
                        av[h][q][t] = *pa[t];
                        pa[t] += step;
                    }
                }
            };
            // one stage's loads in flight under the other's products (c0 is a
            // multiple of two stages)
            static_assert(CHB % (8 * KS) == 0, "whole pairs of stages");
            if(c0 > 0) // uniform
                load(0);
#pragma unroll 1
            for(int k0 = 0; k0 < c0; k0 += 8 * KS)
            {
#pragma unroll
                for(int h = 0; h < 2; ++h)
                {
                    if(h == 0 || k0 + 8 * KS < c0) // uniform
                        load(h ^ 1);
#pragma unroll
                    for(int q = 0; q < KS; ++q)
#pragma unroll
                        for(int t = 0; t < CHR; ++t)
#pragma unroll
                            for(int ct = 0; ct < 2; ++ct)
                                acc[t][ct] = M::run(bv[h][q][ct], -av[h][q][t], acc[t][ct]);
                }
            }

            // ---- 2. the diagonal block (rows c0 .. c0+31): to LDS, factored
            // by the first wavefront, row c0 + lane in its lanes 0 .. jb-1
            if(g0 == 0) // uniform
            {
                const int wl = fresh_tid() & 63;
#pragma unroll
                for(int t = 0; t < (NW == 1 ? 2 : 1); ++t)
                    if(wid + t * NW < 2)
#pragma unroll
                        for(int ct = 0; ct < 2; ++ct)
#pragma unroll
                            for(int r = 0; r < 4; ++r)
                                sX[wid + t * NW][(wl & 15) * TS + 16 * ct + M::row(wl, r)]
                                    = acc[t][ct][r];
                __syncthreads();
                if(wid == 0)
                {
                    // lane = row + 32 h holds columns 2 q + h of its row; the
                    // finished column k reaches the lanes through LDS.
                    // Entries above the diagonal and past jb are never used.
                    const int fl = fresh_tid() & 63;
                    const int i = fl & (CHB - 1), h = fl >> 5;
                    T d[CHB / 2];
#pragma unroll
                    for(int q = 0; q < CHB / 2; ++q)
                        d[q] = sX[i >> 4][(i & 15) * TS + 2 * q + h];
#pragma unroll
                    for(int k = 0; k < CHB; ++k)
                    {
                        int ik = i; // one column's masks at a time
                        asm volatile("" : "+v"(ik));
                        const T t = readlane_t(d[k / 2], k + CHB * (k & 1)); // updated a_kk
                        // columns past jb hold copies: factored, never stored
                        const bool bad = t <= T(0); // uniform
                        if(bad && k < jb && fl == 0 && sinfo == 0)
                            sinfo = c0 + k + 1;
                        const T root = sqrt_t(t);
                        const T piv = bad ? t : root;
                        const T r = bad ? T(0) : T(1) / root;
                        const T l = ik == k ? piv : d[k / 2] * r;
                        if(h == (k & 1) && ik >= k)
                        {
                            d[k / 2] = l;
                            sL11[k * CHB + ik] = l;
                        }
                        if(fl == 0)
                            sres[k] = r;
                        wave_sync();
                        // trailing entries: a_jm -= l_jk l_mk, m in (k, j]
                        const T* col = sL11 + k * CHB + after(d);
                        const T lik = col[ik];
#pragma unroll
                        for(int q = k / 2; q < CHB / 2; ++q)
                            if(2 * q + 1 > k)
                            {
                                const T z = fma_t(-lik, col[2 * q + h], d[q]);
                                if(2 * q > k)
                                    d[q] = z;
                                else
                                    d[q] = h ? z : d[q];
                            }
                    }
#pragma unroll
                    for(int q = 0; q < CHB / 2; ++q)
                        if(2 * q + h <= i && i < jb)
                            L(c0 + i, c0 + 2 * q + h) = d[q];
                }
                __syncthreads();
            }

            // ---- 3. rows below the diagonal block, 16 at a time through LDS
            // to four lanes per row
            T* sx = sX[wid];
#pragma unroll
            for(int t = 0; t < CHR; ++t)
            {
                const int lane = fresh_tid() & 63;
                const int i0 = c0 + 16 * (g0 + wid + t * NW);
                if(i0 >= c0 + CHB && i0 < n) // uniform in the wavefront
                {
                    wave_sync();
#pragma unroll
                    for(int ct = 0; ct < 2; ++ct)
#pragma unroll
                        for(int r = 0; r < 4; ++r)
                            sx[(lane & 15) * TS + 16 * ct + M::row(lane, r)] = acc[t][ct][r];
                    wave_sync();
                    T x[CHB / 4];
#pragma unroll
                    for(int q = 0; q < CHB / 4; ++q)
                        x[q] = sx[(lane >> 2) * TS + 4 * q + (lane & 3)];
                    chol_row_solve<T>(sL11, sres, lane, x);
                    const int i = i0 + (lane >> 2);
                    if(i < n)
                    {
#pragma unroll
                        for(int q = 0; q < CHB / 4; ++q)
                            L(i, c0 + 4 * q + (lane & 3)) = x[q];
                    }
                }
            }
        }
        __syncthreads(); // the block column is written before the next one reads it
    }
    if(tid == 0)
        info[b] = sinfo;
}

// One system and 16 right-hand sides per workgroup (n <= NMAX): the two
// non-unit triangular solves with the factor.  skip[b] != 0: B of system b is
// left unchanged (posv after a failed factorisation).
template <typename T, int NMAX, int NT, bool UP>
__global__ __launch_bounds__(NT, (tile_waves<T, NMAX, NT>())) void potrs_fused_kernel(
    int n, int nrhs, Batch<T> AA, int lda, Batch<T> BB, int ldb, int bc, unsigned chunks,
    unsigned chunk0, const int* __restrict__ skip)
{
    unsigned chunk;
    const int64_t b = tile_solve_system(blockIdx.x, chunks, chunk);
    if(b >= bc || (skip && skip[b] != 0))
        return;
    const int c0 = int(chunk0 + chunk) * TSC;
    const int cend = nrhs - c0 < TSC ? nrhs : c0 + TSC;
    tile_solve_body<T, NMAX, NT, UP ? TILE_CHOL_U : TILE_CHOL_L, false>(
        n, c0, cend, AA[b], lda, nullptr, BB[b], ldb, BB[b], ldb);
}

// The same by rows (blockDim.x == NMAX, n <= NMAX, nrhs <= NR).
template <typename T, int NMAX, int NR, bool UP>
__global__ __launch_bounds__(NMAX) void potrs_rows_kernel(int n, int nrhs, Batch<T> AA, int lda,
                                                          Batch<T> BB, int ldb,
                                                          const int* __restrict__ skip)
{
    __shared__ T sx[2][GBS][NR];
    __shared__ T sL[GBS][GBS + 1];
    const int64_t b = blockIdx.x;
    if(skip && skip[b] != 0)
        return;
    const int tid = threadIdx.x;
    const MatrixBuffer<T> A(AA[b], lda, n);
    T* Bm = BB[b];
    const MatrixBuffer<T> Bbuf(Bm, ldb, nrhs);
    T x[NR];
#pragma unroll
    for(int q = 0; q < NR; ++q)
        x[q] = Bbuf.load(tid < n && q < nrhs ? Bbuf.row_offset(tid) + Bbuf.col_offset(q)
                                             : MatrixBuffer<T>::OUT_OF_RANGE,
                         0);
    solve_lower_rows<T, NR, UP, false, true>(n, A, x, sx, sL); // L or U^T
    solve_upper_rows<T, NR, !UP, false, true>(n, A, x, sx, sL); // L^T or U
    if(tid < n)
    {
#pragma unroll
        for(int q = 0; q < NR; ++q)
            if(q < nrhs)
                Bm[tid + int64_t(q) * ldb] = x[q];
    }
}

// Any order: one thread per (system, right-hand side), column-oriented
// substitution in the same order of operations.
template <typename T>
__global__ __launch_bounds__(64) void potrs_serial_kernel(int n, int nrhs, Batch<T> AA, int lda,
                                                          int up, Batch<T> BB, int ldb, int bc,
                                                          int64_t block0,
                                                          const int* __restrict__ skip)
{
    const int64_t g = (block0 + blockIdx.x) * blockDim.x + threadIdx.x;
    if(g >= int64_t(bc) * nrhs)
        return;
    const int64_t b = g / nrhs;
    const int c = int(g % nrhs);
    if(skip && skip[b] != 0)
        return;
    const T* A = AA[b];
    auto L = [&](int i, int j) { return up ? A[j + int64_t(i) * lda] : A[i + int64_t(j) * lda]; };
    T* x = BB[b] + int64_t(c) * ldb;
    for(int k = 0; k < n; ++k)
    {
        x[k] = x[k] / L(k, k);
        for(int i = k + 1; i < n; ++i)
            x[i] = fma_t(-L(i, k), x[k], x[i]);
    }
    for(int k = n - 1; k >= 0; --k)
    {
        x[k] = x[k] / L(k, k);
        for(int i = 0; i < k; ++i)
            x[i] = fma_t(-L(k, i), x[k], x[i]);
    }
}

template <typename T>
rocblas_status potrf(hipStream_t stream, bool up, int n, Batch<T> A, int lda, int* info, int bc)
{
    if(bc <= 0)
        return rocblas_status_success;
    if(n <= 0)
        return reset_info(stream, info, bc);
    auto go = [&](auto nt) {
        constexpr int NT = decltype(nt)::value;
        return launch_split(bc, 1, NT, 1, [&](int64_t b0, int64_t nb, int64_t, int64_t) {
            const dim3 grid{unsigned(nb)};
            if(up)
                hipLaunchKernelGGL((potrf_kernel<T, NT, true>), grid, dim3(NT), 0, stream, n,
                                   batch_from(A, b0), lda, info + b0);
            else
                hipLaunchKernelGGL((potrf_kernel<T, NT, false>), grid, dim3(NT), 0, stream, n,
                                   batch_from(A, b0), lda, info + b0);
            RSA_LAUNCH_CHECK();
            return rocblas_status_success;
        });
    };
    // as many wavefronts as the first block column gives 16-row groups
    if(n <= 64)
        return go(std::integral_constant<int, 64>{});
    if(n <= 128)
        return go(std::integral_constant<int, 128>{});
    return go(std::integral_constant<int, 256>{});
}

template <typename T>
rocblas_status potrs(hipStream_t stream, bool up, int n, int nrhs, Batch<T> A, int lda,
                     Batch<T> B, int ldb, int bc, const int* skip)
{
    if(bc <= 0 || n <= 0 || nrhs <= 0)
        return rocblas_status_success;
    using std::integral_constant;
    if(n <= FUSED_MAX && fits_buffer<T>(lda, n) && fits_buffer<T>(ldb, nrhs))
    {
        if(potrs_by_rows<T>(n, nrhs, bc))
        {
            auto rows = [&](auto nmax, auto nr) {
                constexpr int NMAX = decltype(nmax)::value;
                constexpr int NR = decltype(nr)::value;
                return launch_split(bc, 1, NMAX, 1, [&](int64_t b0, int64_t nb, int64_t, int64_t) {
                    const dim3 grid{unsigned(nb)};
                    const int* sk = skip ? skip + b0 : nullptr;
                    if(up)
                        hipLaunchKernelGGL((potrs_rows_kernel<T, NMAX, NR, true>), grid, dim3(NMAX),
                                           0, stream, n, nrhs, batch_from(A, b0), lda,
                                           batch_from(B, b0), ldb, sk);
                    else
                        hipLaunchKernelGGL((potrs_rows_kernel<T, NMAX, NR, false>), grid,
                                           dim3(NMAX), 0, stream, n, nrhs, batch_from(A, b0), lda,
                                           batch_from(B, b0), ldb, sk);
                    RSA_LAUNCH_CHECK();
                    return rocblas_status_success;
                });
            };
            auto by_nrhs = [&](auto nmax) {
                return nrhs == 1 ? rows(nmax, integral_constant<int, 1>{})
                                 : rows(nmax, integral_constant<int, 4>{});
            };
            // the orders and right-hand sides that potrs_by_rows can give
            if(n <= 64)
                return nrhs <= 4 ? by_nrhs(integral_constant<int, 64>{})
                                 : rows(integral_constant<int, 64>{}, integral_constant<int, 8>{});
            if(n <= 128)
                return by_nrhs(integral_constant<int, 128>{});
            if(n <= 256 || sizeof(T) == 4)
                return by_nrhs(integral_constant<int, 256>{});
            if constexpr(sizeof(T) == 8)
                return by_nrhs(integral_constant<int, 512>{});
        }
        auto go = [&](auto nmax, auto nt) {
            constexpr int NMAX = decltype(nmax)::value;
            constexpr int NT = decltype(nt)::value;
            return launch_split(
                bc, ceil_div(nrhs, TSC), NT, TILE_XCDS,
                [&](int64_t b0, int64_t nb, int64_t c0, int64_t nc) {
                    const dim3 grid{unsigned(tile_solve_grid(int(nb), int(nc)))};
                    const int* sk = skip ? skip + b0 : nullptr;
                    if(up)
                        hipLaunchKernelGGL((potrs_fused_kernel<T, NMAX, NT, true>), grid, dim3(NT),
                                           0, stream, n, nrhs, batch_from(A, b0), lda,
                                           batch_from(B, b0), ldb, int(nb), unsigned(nc),
                                           unsigned(c0), sk);
                    else
                        hipLaunchKernelGGL((potrs_fused_kernel<T, NMAX, NT, false>), grid, dim3(NT),
                                           0, stream, n, nrhs, batch_from(A, b0), lda,
                                           batch_from(B, b0), ldb, int(nb), unsigned(nc),
                                           unsigned(c0), sk);
                    RSA_LAUNCH_CHECK();
                    return rocblas_status_success;
                });
        };
        constexpr int F = sizeof(T) == 8 ? 2 : 1; // as getrs_fused_launch
        if(n <= 64)
            return go(integral_constant<int, 64>{}, integral_constant<int, 64 * F>{});
        if(n <= 128)
            return go(integral_constant<int, 128>{}, integral_constant<int, 128 * F>{});
        if(n <= 256)
            return go(integral_constant<int, 256>{}, integral_constant<int, 256 * F>{});
        return go(integral_constant<int, 512>{}, integral_constant<int, 512>{});
    }
    return launch_split(
        (int64_t(bc) * nrhs + 63) / 64, 1, 64, 1, [&](int64_t w0, int64_t nw, int64_t, int64_t) {
            hipLaunchKernelGGL((potrs_serial_kernel<T>), dim3(unsigned(nw)), dim3(64), 0, stream, n,
                               nrhs, A, lda, int(up), B, ldb, bc, w0, skip);
            RSA_LAUNCH_CHECK();
            return rocblas_status_success;
        });
}

#define RSA_CHOL_INST(T)                                                                      \
    template rocblas_status potrf<T>(hipStream_t, bool, int, Batch<T>, int, int*, int);       \
    template rocblas_status potrs<T>(hipStream_t, bool, int, int, Batch<T>, int, Batch<T>, int, \
                                     int, const int*);
RSA_CHOL_INST(float)
RSA_CHOL_INST(double)

} // namespace rsa
