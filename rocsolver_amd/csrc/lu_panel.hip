// lu_panel.hip -- register-resident panel of the blocked LU.
//
// One workgroup per matrix holds the W columns A[j0:m, j0:j0+jb] of a panel
// in registers, R rows per thread, and factors them with partial pivoting
// with one barrier per column, as the panel of the fused LU does: every
// wavefront publishes its best candidate row with its key, each thread then
// finds the winner among the wavefronts, and the interchange moves labels
// (the logical row a register row holds), not data.  The rows are written
// back once, to their final positions.  Interchange semantics: the same final
// rows as roclapack_getf2.hpp:41-99.
//
// The kernel then applies the panel's interchanges to the other columns of
// [o0, oend) and solves U12 = L11^-1 A12 for those right of the panel.
//
// What bounds it: the chain of dependent column steps (arg-max across the
// workgroup, broadcast of the winning row, rank-1 update of R rows a thread).
// Reading and writing the panel in global memory at every column, with two
// barriers, took 303 us for a 32-column FP64 panel of n = 1024 on average
// (64 matrices); this kernel takes 76 us there.
#include "internal.hpp"

#include <climits>

namespace rsa
{

// largest / smallest over groups of NW (4 or 8) consecutive lanes
template <int NW, typename I>
__device__ __forceinline__ I few_max(I v)
{
    auto mx = [](I a, I b) { return a > b ? a : b; };
    v = mx(v, I(dpp_mov<0xB1>(int(v))));
    v = mx(v, I(dpp_mov<0x4E>(int(v))));
    if(NW == 8)
        v = mx(v, I(dpp_mov<0x141>(int(v))));
    return v;
}
template <int NW>
__device__ __forceinline__ int few_min(int v)
{
    v = min(v, dpp_mov<0xB1>(v));
    v = min(v, dpp_mov<0x4E>(v));
    if(NW == 8)
        v = min(v, dpp_mov<0x141>(v));
    return v;
}

// Index of the largest key among NW candidates, one per lane of each group of
// NW lanes (a negative key: no candidate), ties to the smaller index; at
// least one is a candidate.  As group_argmax, on the bit patterns.
template <int NW>
__device__ __forceinline__ int few_argmax(double key, int idx)
{
    const bool cand = key >= 0.0;
    const uint64_t u = cand ? uint64_t(__double_as_longlong(key)) : 0u;
    const int hi = int(u >> 32);
    const unsigned lo = unsigned(u);
    const int mh = few_max<NW>(hi);
    const unsigned ml = few_max<NW>(hi == mh ? lo : 0u);
    return few_min<NW>((cand && hi == mh && lo == ml) ? idx : 0x7fffffff);
}
template <int NW>
__device__ __forceinline__ int few_argmax(float key, int idx)
{
    const bool cand = key >= 0.f;
    const int u = cand ? __float_as_int(key) : 0;
    const int mu = few_max<NW>(u);
    return few_min<NW>((cand && u == mu) ? idx : 0x7fffffff);
}

// m - j0 <= R * NT rows, jb <= W columns; W * lda * sizeof(T) below 2^31.
// Row indices inside the kernel count from j0.
template <typename T, int W, int R, int NT, bool PIVOT>
__global__ __launch_bounds__(NT, 2) void panel_reg_kernel(int m, Batch<T> AA, int lda,
                                                          int* __restrict__ ipivA, int64_t strideP,
                                                          int* __restrict__ info, int j0, int jb,
                                                          int o0, int oend)
{
    constexpr int NW = NT / 64;
    constexpr int G = 16 / int(sizeof(T)); // entries per 16-byte group
    constexpr int CH = 8; // columns of the pivot row read at a time
    static_assert((NW == 4 || NW == 8) && W % CH == 0 && 2 * W <= 64, "panel shape");
    typedef T g16_t __attribute__((ext_vector_type(G)));
    __shared__ __align__(16) T scand[2][NW][W];
    __shared__ T skey[2][NW];
    __shared__ int slab[2][NW];
    __shared__ __align__(16) T sL[W * W]; // L11 by columns
    __shared__ int s_swap[W]; // row interchanged with row k (itself: none)
    __shared__ int s_pos[2 * W]; // rows touched by the interchanges
    __shared__ int s_src[2 * W]; // row whose entries end at s_pos[q]
    __shared__ int s_cnt;

    const int64_t b = blockIdx.x;
    T* A = AA[b] + j0;
    const int tid = threadIdx.x;
    const int wid = tid / 64;
    const int lane = tid % 64;
    const int mp = m - j0;
    const MatrixBuffer<T> P(A + int64_t(j0) * lda, lda, jb);

    T v[R][W];
    int label[R]; // logical row of each register row, -1 past the last
#pragma unroll
    for(int r = 0; r < R; ++r)
    {
        const int i = tid + r * NT;
        const bool act = i < mp;
        label[r] = act ? i : -1;
        uint32_t off = P.offset(act, i, 0);
        const uint32_t step = act ? P.ld_bytes : 0u;
#pragma unroll
        for(int q = 0; q < W; ++q)
        {
            v[r][q] = P.load(off, 0); // 0 past column jb
            off += step;
            opaque(off);
        }
    }

    int zero_at = 0;
#pragma unroll
    for(int k = 0; k < W; ++k)
    {
        if(k < jb) // uniform
        {
            const int par = k & 1;
            T key = T(-1);
            int lab = INT_MAX;
            if(PIVOT)
            {
#pragma unroll
                for(int r = 0; r < R; ++r)
                {
                    const T kk = label[r] >= k ? pivot_key(v[r][k], label[r] == k) : T(-1);
                    const bool better = (kk > key) | ((kk == key) & (label[r] < lab) & (kk >= T(0)));
                    key = better ? kk : key;
                    lab = better ? label[r] : lab;
                }
                wave_argmax(key, lab);
            }
            else
                lab = k;
            // the row held by this wavefront that may become the pivot row
            // (whole 16-byte groups from the one holding column k)
#pragma unroll
            for(int r = 0; r < R; ++r)
                if(label[r] == lab)
                {
                    const int at = PIVOT ? wid : 0;
#pragma unroll
                    for(int j = 0; j < W; ++j)
                        if(j / G >= k / G)
                            scand[par][at][j] = v[r][j];
                }
            if(PIVOT && lane == 0)
            {
                skey[par][wid] = key;
                slab[par][wid] = lab;
            }
            __syncthreads();
            int bl = k, wb = 0;
            if(PIVOT)
            {
                const int cw = lane & (NW - 1);
                const T ck = skey[par][cw];
                const int cl = slab[par][cw];
                const int best = few_argmax<NW>(ck, (cl << 3) | cw);
                bl = __builtin_amdgcn_readfirstlane(best >> 3);
                wb = best & 7;
            }
            const T* prow = &scand[par][0][0] + wb * W;
            const T pv = prow[k];
            const bool nz = pv != T(0);
            // a zero pivot leaves the column alone with pivoting (every
            // candidate is zero) and multiplies it by zero without (the
            // reference npvt kernels keep the scale at 0:
            // roclapack_getf2_specialized_kernels.hpp:185-188,427-430)
            const T rcp = nz ? T(1) / pv : T(0);
            if(!nz && zero_at == 0)
                zero_at = k + 1;
            if(PIVOT && tid == 0)
                s_swap[k] = bl;
            bool below[R];
            T l[R];
#pragma unroll
            for(int r = 0; r < R; ++r)
            {
                if(PIVOT)
                    label[r] = label[r] == bl ? k : (label[r] == k ? bl : label[r]);
                below[r] = label[r] > k;
                l[r] = v[r][k];
                if(nz || !PIVOT)
                    l[r] *= rcp;
                v[r][k] = below[r] ? l[r] : v[r][k];
            }
#pragma unroll
            for(int c8 = (k + 1) / CH * CH; c8 < W; c8 += CH)
            {
                T u[CH];
#pragma unroll
                for(int g = 0; g < CH / G; ++g)
                {
                    if(c8 + g * G + G - 1 > k)
                    {
                        const g16_t t = *reinterpret_cast<const g16_t*>(prow + c8 + g * G);
#pragma unroll
                        for(int e = 0; e < G; ++e)
                            u[g * G + e] = t[e];
                    }
                }
#pragma unroll
                for(int r = 0; r < R; ++r)
                    if(below[r])
                    {
#pragma unroll
                        for(int q = 0; q < CH; ++q)
                            if(c8 + q > k)
                                v[r][c8 + q] = fma_t(-l[r], u[q], v[r][c8 + q]);
                    }
            }
        }
    }

    __syncthreads(); // s_swap is complete

    // rows back to their final positions, L11 to LDS
#pragma unroll
    for(int r = 0; r < R; ++r)
    {
        const bool act = label[r] >= 0;
        uint32_t off = P.offset(act, label[r], 0);
        const uint32_t step = act ? P.ld_bytes : 0u;
#pragma unroll
        for(int q = 0; q < W; ++q)
        {
            P.store(v[r][q], off, 0); // columns past jb are dropped
            off += step;
            opaque(off);
        }
        if(act && label[r] < W)
        {
#pragma unroll
            for(int q = 0; q < W; ++q)
                sL[q * W + label[r]] = v[r][q];
        }
    }
    if(tid == 0 && zero_at != 0 && info[b] == 0)
        info[b] = j0 + zero_at;
    if(PIVOT && tid < jb)
        ipivA[b * strideP + j0 + tid] = j0 + s_swap[tid] + 1;

    const int nout = oend - o0 - jb; // the other columns of [o0, oend)
    if(nout <= 0) // uniform
        return;
    if(PIVOT)
    {
        // the interchanges composed into one map of at most 2 jb rows: lane q
        // of the first wavefront keeps slot q (row pos, source src); ballots
        // find a row's slot, a new row takes the next free one
        if(wid == 0)
        {
            int pos = -1, src = -1, cnt = 0;
            for(int k = 0; k < jb; ++k)
            {
                const int r2 = __builtin_amdgcn_readfirstlane(s_swap[k]);
                if(r2 == k) // uniform
                    continue;
                int qs[2];
#pragma unroll
                for(int h = 0; h < 2; ++h)
                {
                    const int row = h ? r2 : k;
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
        // one wavefront per column, lane q moving the entry of slot q; the
        // loads of four columns in flight
        const bool mine = lane < s_cnt;
        const int pos = mine ? s_pos[lane] : 0, src = mine ? s_src[lane] : 0;
        constexpr int UC = 4;
        for(int e0 = wid * UC; e0 < nout; e0 += NW * UC)
        {
            T x[UC];
#pragma unroll
            for(int u = 0; u < UC; ++u)
            {
                const int j = o0 + e0 + u < j0 ? o0 + e0 + u : o0 + e0 + u + jb;
                x[u] = (mine && e0 + u < nout) ? A[src + int64_t(j) * lda] : T(0);
            }
#pragma unroll
            for(int u = 0; u < UC; ++u)
            {
                const int j = o0 + e0 + u < j0 ? o0 + e0 + u : o0 + e0 + u + jb;
                if(mine && e0 + u < nout)
                    A[pos + int64_t(j) * lda] = x[u];
            }
        }
    }
    __syncthreads(); // the interchanged rows are written, L11 is in LDS

    // U12 = L11^-1 A12, one thread per column.  L11 is read through an offset
    // that the optimiser must take as computed from x[k] every two columns
    // (an empty asm tied to x[k]), so its entries are not all loaded ahead of
    // the substitution (and spilled).
    for(int j = j0 + jb + tid; j < oend; j += NT)
    {
        T* col = A + int64_t(j) * lda;
        T x[W];
#pragma unroll
        for(int i = 0; i < W; ++i)
            x[i] = i < jb ? col[i] : T(0);
        const T* L = sL;
#pragma unroll
        for(int k = 0; k < W; ++k)
        {
            if(k < jb) // uniform
            {
                if((k & 1) == 0)
                {
                    uint32_t lo = 0;
                    asm volatile("" : "+v"(lo) : "v"(x[k]));
                    L = sL + lo;
                }
#pragma unroll
                for(int i = k + 1; i < W; ++i)
                    x[i] = fma_t(-L[i + k * W], x[k], x[i]);
            }
        }
#pragma unroll
        for(int i = 0; i < W; ++i)
            if(i < jb)
                col[i] = x[i];
    }
}

// Panel width for `rows` rows: the register file of one CU holds 512 threads
// x 128 (64-bit: 64) values of a panel beside the working set, so the panel
// narrows as it gets taller; 0: too tall (or too long a leading dimension for
// the 32-bit offsets), the caller uses its panel in global memory.
template <typename T>
int panel_reg_width(int rows, int lda)
{
    if(!fits_buffer<T>(lda, 32))
        return 0;
    const int unit = sizeof(T) == 8 ? 1024 : 2048;
    return rows <= unit ? 32 : rows <= 2 * unit ? 16 : rows <= 4 * unit ? 8 : 0;
}

template <typename T>
rocblas_status panel_reg(hipStream_t stream, int m, Batch<T> A, int lda, int* ipiv,
                         int64_t strideP, int* info, int j0, int jb, int o0, int oend, int bc,
                         bool pivot)
{
    auto go = [&](auto w, auto r, auto nt) {
        constexpr int W = decltype(w)::value;
        constexpr int R = decltype(r)::value;
        constexpr int NT = decltype(nt)::value;
        if(pivot)
            hipLaunchKernelGGL((panel_reg_kernel<T, W, R, NT, true>), dim3(bc), dim3(NT), 0, stream,
                               m, A, lda, ipiv, strideP, info, j0, jb, o0, oend);
        else
            hipLaunchKernelGGL((panel_reg_kernel<T, W, R, NT, false>), dim3(bc), dim3(NT), 0,
                               stream, m, A, lda, ipiv, strideP, info, j0, jb, o0, oend);
    };
    using std::integral_constant;
    constexpr int S = sizeof(T) == 8 ? 1 : 2;
    const int rows = m - j0;
    if(rows <= 256)
        go(integral_constant<int, 32>{}, integral_constant<int, 1>{}, integral_constant<int, 256>{});
    else if(rows <= 512)
        go(integral_constant<int, 32>{}, integral_constant<int, 1>{}, integral_constant<int, 512>{});
    else if(rows <= 1024)
        go(integral_constant<int, 32>{}, integral_constant<int, 2>{}, integral_constant<int, 512>{});
    else if(rows <= 2048)
        go(integral_constant<int, 16 * S>{}, integral_constant<int, 4>{},
           integral_constant<int, 512>{});
    else if(rows <= 4096)
        go(integral_constant<int, 8 * S>{}, integral_constant<int, 8>{},
           integral_constant<int, 512>{});
    else if constexpr(sizeof(T) == 4)
        go(integral_constant<int, 8>{}, integral_constant<int, 16>{}, integral_constant<int, 512>{});
    RSA_LAUNCH_CHECK();
    return rocblas_status_success;
}

#define RSA_PANEL_INST(T)                                                                       \
    template int panel_reg_width<T>(int, int);                                                  \
    template rocblas_status panel_reg<T>(hipStream_t, int, Batch<T>, int, int*, int64_t, int*,  \
                                         int, int, int, int, int, bool);
RSA_PANEL_INST(float)
RSA_PANEL_INST(double)

} // namespace rsa
