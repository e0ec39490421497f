// lu_panel.hip -- register-resident panel of the blocked LU.
//
// One workgroup per matrix holds the W columns A[j0:m, j0:j0+jb] of a panel
// in registers, R rows per thread, and factors them with partial pivoting, as
// the panel of the fused LU does (pivot_step.hpp): every wavefront publishes
// its best candidate, each thread then finds the winner among them, the
// winner's row goes to LDS, and the interchange moves labels (the logical row
// a register row holds), not data.  The rows are written
// back once, to their final positions.  Interchange semantics: the same final
// rows as roclapack_getf2.hpp:41-99.
//
// The kernel then applies the panel's interchanges to the other columns of
// [o0, oend) and solves U12 = L11^-1 A12 for those right of the panel up to
// uend.
//
// What bounds it: the chain of dependent column steps (arg-max across the
// workgroup, broadcast of the winning row, rank-1 update of R rows a thread).
// Reading and writing the panel in global memory at every column, with two
// barriers, took 303 us for a 32-column FP64 panel of n = 1024 on average
// (64 matrices); this kernel takes 40 us there.
#include "internal.hpp"
#include "mfma.hpp"
#include "pivot_step.hpp"
#include "quad_solve.hpp"

#include <climits>

namespace rsa
{

// m - j0 <= R * NT rows, jb <= W columns; W * lda * sizeof(T) below 2^31.
// Row indices inside the kernel count from j0.
template <typename T, int W, int R, int NT, bool PIVOT>
__global__ __launch_bounds__(NT, 2) void panel_reg_kernel(int m, Batch<T> AA, int lda,
                                                          int* __restrict__ ipivA, int64_t strideP,
                                                          int* __restrict__ info, int j0, int jb,
                                                          int o0, int oend, int uend)
{
    constexpr int NW = NT / 64;
    constexpr int G = 16 / int(sizeof(T)); // entries per 16-byte group
    constexpr int CH = 8; // columns of the pivot row read at a time
    static_assert((NW == 4 || NW == 8) && W % CH == 0 && 2 * W <= 64, "panel shape");
    typedef T g16_t __attribute__((ext_vector_type(G)));
    __shared__ __align__(16) T srow[2][W]; // pivot row
    __shared__ PivotRecord srec[2][NW];
    __shared__ __align__(16) T sL[W * W]; // L11 by columns
    __shared__ int s_swap[W]; // row interchanged with row k (itself: none)

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
            int bl = k, wave = 0;
            T pv, rcp;
            if(PIVOT)
            {
                T key = T(-1), val = T(0);
                int lab = INT_MAX;
#pragma unroll
                for(int r = 0; r < R; ++r)
                {
                    const T kk = label[r] >= k ? pivot_key(v[r][k], label[r] == k) : T(-1);
                    const bool better = (kk > key) | ((kk == key) & (label[r] < lab) & (kk >= T(0)));
                    key = better ? kk : key;
                    lab = better ? label[r] : lab;
                    val = better ? v[r][k] : val;
                }
                publish_candidate(key, val, lab, &srec[par][wid]);
                __syncthreads();
                select_candidate<T, NW>(srec[par], bl, wave, pv, rcp);
            }
            // the pivot row to LDS (whole 16-byte groups from the one holding
            // column k): only by the thread that holds it, after the choice
            // -- every wavefront's candidate row before it would fill the LDS
            // pipeline, which takes a one-lane 16-byte store as a full one
#pragma unroll
            for(int r = 0; r < R; ++r)
                if(label[r] == bl)
#pragma unroll
                    for(int j = 0; j < W; ++j)
                        if(j / G >= k / G)
                            srow[par][j] = v[r][j];
            __syncthreads();
            const T* prow = srow[par];
            if(PIVOT)
            {
                pv = readlane_t(pv, wave);
                rcp = readlane_t(rcp, wave);
            }
            else
            {
                pv = prow[k];
                rcp = T(1) / pv;
            }
            const bool nz = pv != T(0);
            // a zero pivot leaves the column alone with pivoting (every
            // candidate is zero) and multiplies it by zero without (the
            // reference npvt kernels keep the scale at 0:
            // roclapack_getf2_specialized_kernels.hpp:185-188,427-430)
            rcp = nz ? rcp : T(0);
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
        // follows row q, lane W + q the row that row q was interchanged with,
        // back through the interchanges to where its entries are now
        const int q = lane & (2 * W - 1);
        const int pos = q < W ? q : (q - W < jb ? s_swap[q - W] : -1);
        int src = pos;
        for(int k = jb - 1; k >= 0; --k)
        {
            const int p = s_swap[k];
            src = src == k ? p : (src == p ? k : src);
        }
        // rows of the second half below jb are in the first; a row met twice
        // there is moved twice, the same entry to the same place
        const bool mine = (q < W ? q < jb : pos >= jb) && src != pos;
        // 64 / (2 W) columns per wavefront, the loads of four such groups in
        // flight
        constexpr int UC = 4, CPW = 64 / (2 * W);
        for(int e0 = wid * UC * CPW + lane / (2 * W); e0 < nout; e0 += NW * UC * CPW)
        {
            T x[UC];
            auto at = [&](int row, int u) -> T& {
                const int e = o0 + e0 + u * CPW;
                return A[row + int64_t(e < j0 ? e : e + jb) * lda];
            };
#pragma unroll
            for(int u = 0; u < UC; ++u)
                x[u] = (mine && e0 + u * CPW < nout) ? at(src, u) : T(0);
#pragma unroll
            for(int u = 0; u < UC; ++u)
                if(mine && e0 + u * CPW < nout)
                    at(pos, u) = x[u];
        }
    }
    __syncthreads(); // the interchanged rows are written, L11 is in LDS

    // U12 = L11^-1 A12, four lanes per column
    for(int j = j0 + jb + tid / 4; j < uend; j += NT / 4)
    {
        T* col = A + int64_t(j) * lda + (lane & 3);
        T x[W / 4];
#pragma unroll
        for(int t = 0; t < W / 4; ++t)
            x[t] = 4 * t + (lane & 3) < jb ? col[4 * t] : T(0);
        quad_solve<T, W, true, true>(sL, lane, x);
#pragma unroll
        for(int t = 0; t < W / 4; ++t)
            if(4 * t + (lane & 3) < jb)
                col[4 * t] = x[t];
    }
}

// ------------------------------------------------------------ outer block
// The finished block column [o0, o0 + nb), nb <= OUTER_NB, applied to the
// columns outside it: its interchanges to all of them, and U12 = L11^-1 A12
// for those right of it.  64 columns per workgroup; the left_chunks first
// workgroups of a matrix take the columns left of the block.
//
// Bound by latency and by the scattered rows of the interchanges (one cache
// line per row and column), so one block's interchanges are composed into a
// map and applied once, not panel by panel.  The nb top rows stay in LDS from
// the interchange to the solve: diagonal blocks of DB rows by substitution (four
// lanes per column), the rows below by matrix-core products.  Each wavefront
// owns 16 columns from then on, so the solve has no barrier.
constexpr int OUTER_COLS = 64;

template <typename T, bool PIVOT, int DB>
__global__ __launch_bounds__(256, 1) void outer_apply_kernel(int n, Batch<T> AA, int lda,
                                                             const int* __restrict__ ipivA,
                                                             int64_t strideP, int o0, int nb,
                                                             int left_chunks, int64_t boff)
{
    using M = mfma16<T>;
    constexpr int LS = OUTER_NB + 1; // column stride of the right-hand sides in LDS
    constexpr int UC = 16; // columns in flight
    __shared__ T sB[OUTER_COLS * LS];
    __shared__ __align__(16) T sL[OUTER_NB / DB][DB * DB];
    __shared__ int s_piv[OUTER_NB];

    const int64_t b = blockIdx.y + boff;
    T* A = AA[b] + o0;
    const int tid = threadIdx.x;
    const int wid = tid / 64;
    const int lane = tid % 64;
    const int chunk = blockIdx.x;
    const bool right = chunk >= left_chunks; // uniform
    const int c0 = right ? o0 + nb + (chunk - left_chunks) * OUTER_COLS : chunk * OUTER_COLS;
    const int nc = (right ? n : o0) - c0 < OUTER_COLS ? (right ? n : o0) - c0 : OUTER_COLS;

    if(PIVOT && tid < nb)
        s_piv[tid] = ipivA[b * strideP + o0 + tid] - 1 - o0;
    if(right)
    {
#pragma unroll
        for(int d = 0; d < OUTER_NB / DB; ++d)
            for(int e = tid; e < DB * DB; e += 256)
            {
                const int i = DB * d + e % DB, k = DB * d + e / DB;
                sL[d][e] = (i < nb && k < nb) ? A[i + int64_t(o0 + k) * lda] : T(0);
            }
    }
    __syncthreads();

    // threads 0..127 follow the rows of the block, threads 128..255 the rows
    // they were interchanged with, back to where their entries are now (a row
    // below the block met twice is moved twice, the same entry to the same
    // place)
    int pos = tid < OUTER_NB ? tid : -1, src = pos;
    if(PIVOT)
    {
        if(tid >= OUTER_NB && tid - OUTER_NB < nb)
            pos = s_piv[tid - OUTER_NB];
        src = pos;
        for(int k = nb - 1; k >= 0; --k)
        {
            const int p = s_piv[k];
            src = src == k ? p : (src == p ? k : src);
        }
    }
    const bool top = tid < OUTER_NB;
    const bool load = top ? (tid < nb && (right || src != pos)) : (pos >= nb && src != pos);
    for(int cb = 0; cb < nc; cb += UC) // uniform
    {
        T x[UC];
#pragma unroll
        for(int u = 0; u < UC; ++u)
            x[u] = (load && cb + u < nc) ? A[src + int64_t(c0 + cb + u) * lda] : T(0);
        __syncthreads(); // the loads of these columns are done
        if(right && top)
        {
#pragma unroll
            for(int u = 0; u < UC; ++u)
                sB[(cb + u) * LS + tid] = x[u];
        }
        else if(load)
        {
#pragma unroll
            for(int u = 0; u < UC; ++u)
                if(cb + u < nc)
                    A[pos + int64_t(c0 + cb + u) * lda] = x[u];
        }
    }
    if(!right)
        return;
    __syncthreads();

    if(16 * wid >= nc) // uniform in the wavefront
        return;
    T* colB = sB + 16 * wid * LS; // this wavefront's 16 columns
#pragma unroll
    for(int d = 0; d < OUTER_NB / DB; ++d)
    {
        if(DB * d < nb) // uniform
        {
            {
                T x[DB / 4];
                T* xp = colB + (lane >> 2) * LS + DB * d + (lane & 3);
#pragma unroll
                for(int t = 0; t < DB / 4; ++t)
                    x[t] = xp[4 * t];
                quad_solve<T, DB, true, true>(sL[d], lane, x);
#pragma unroll
                for(int t = 0; t < DB / 4; ++t)
                    xp[4 * t] = x[t];
            }
            wave_sync();
            // rows below the diagonal block, 16 at a time
            T bv[DB / 4];
#pragma unroll
            for(int ks = 0; ks < DB / 4; ++ks)
                bv[ks] = colB[(lane & 15) * LS + DB * d + 4 * ks + (lane >> 4)];
            for(int i0 = DB * (d + 1); i0 < nb; i0 += 16) // uniform
            {
                const int i = i0 + (lane & 15);
                T av[DB / 4];
#pragma unroll
                for(int ks = 0; ks < DB / 4; ++ks)
                    av[ks] = i < nb ? A[i + int64_t(o0 + DB * d + 4 * ks + (lane >> 4)) * lda]
                                    : T(0);
                typename M::acc_t acc = {0, 0, 0, 0};
#pragma unroll
                for(int ks = 0; ks < DB / 4; ++ks)
                    acc = M::run(av[ks], bv[ks], acc);
#pragma unroll
                for(int r = 0; r < 4; ++r)
                    colB[(lane & 15) * LS + i0 + M::row(lane, r)] -= acc[r];
            }
            wave_sync();
        }
    }
    for(int c = 0; c < 16; ++c)
        if(16 * wid + c < nc) // uniform
            for(int i = lane; i < nb; i += 64)
                A[i + int64_t(c0 + 16 * wid + c) * lda] = colB[c * LS + i];
}

template <typename T>
rocblas_status outer_apply(hipStream_t stream, int n, Batch<T> A, int lda, const int* ipiv,
                           int64_t strideP, int o0, int nb, int bc, bool pivot, int db)
{
    const int left = pivot ? ceil_div(o0, OUTER_COLS) : 0;
    const int chunks = left + ceil_div(n - o0 - nb, OUTER_COLS);
    if(chunks <= 0)
        return rocblas_status_success;
    for(int64_t b0 = 0; b0 < bc; b0 += 65535)
    {
        const int cnt = int((bc - b0) < 65535 ? (bc - b0) : 65535);
        auto go = [&](auto piv, auto d) {
            hipLaunchKernelGGL((outer_apply_kernel<T, decltype(piv)::value, decltype(d)::value>),
                               dim3(chunks, cnt), dim3(256), 0, stream, n, A, lda, ipiv, strideP,
                               o0, nb, left, b0);
        };
        using std::integral_constant;
        if(pivot) // the block column of a matrix
            go(std::true_type{}, integral_constant<int, 32>{});
        else if(db == 8) // part of one: by its panels
            go(std::false_type{}, integral_constant<int, 8>{});
        else if(db == 16)
            go(std::false_type{}, integral_constant<int, 16>{});
        else
            go(std::false_type{}, integral_constant<int, 32>{});
        RSA_LAUNCH_CHECK();
    }
    return rocblas_status_success;
}

// Panel width for `rows` rows: the register file of one CU holds 512 threads
// x 128 values (FP64: 96) of a panel beside the working set, so the panel
// narrows as it gets taller (32 columns of 1025..1536 FP64 rows on three rows
// a thread against 16 on four: n = 2000 5.07 -> 4.92 ms); 0: too tall (or too
// long a leading dimension for the 32-bit offsets), the caller uses its panel
// in global memory.
template <typename T>
int panel_reg_width(int rows, int lda)
{
    if(!fits_buffer<T>(lda, 32))
        return 0;
    if constexpr(sizeof(T) == 8)
        return rows <= 1536 ? 32 : rows <= 2048 ? 16 : rows <= 4096 ? 8 : 0;
    else
        return rows <= 2048 ? 32 : rows <= 4096 ? 16 : rows <= 8192 ? 8 : 0;
}

template <typename T>
rocblas_status panel_reg(hipStream_t stream, int m, Batch<T> A, int lda, int* ipiv,
                         int64_t strideP, int* info, int j0, int jb, int o0, int oend, int uend,
                         int bc, bool pivot)
{
    auto go = [&](auto w, auto r, auto nt) {
        constexpr int W = decltype(w)::value;
        constexpr int R = decltype(r)::value;
        constexpr int NT = decltype(nt)::value;
        return launch_split(bc, 1, NT, 1, [&](int64_t b0, int64_t cnt, int64_t, int64_t) {
            const dim3 grid{unsigned(cnt)};
            int* piv = pivot ? ipiv + b0 * strideP : nullptr;
            if(pivot)
                hipLaunchKernelGGL((panel_reg_kernel<T, W, R, NT, true>), grid, dim3(NT), 0, stream,
                                   m, batch_from(A, b0), lda, piv, strideP, info + b0, j0, jb, o0,
                                   oend, uend);
            else
                hipLaunchKernelGGL((panel_reg_kernel<T, W, R, NT, false>), grid, dim3(NT), 0,
                                   stream, m, batch_from(A, b0), lda, piv, strideP, info + b0, j0,
                                   jb, o0, oend, uend);
            RSA_LAUNCH_CHECK();
            return rocblas_status_success;
        });
    };
    using std::integral_constant;
    constexpr int S = sizeof(T) == 8 ? 1 : 2;
    const int rows = m - j0;
    using i256 = integral_constant<int, 256>;
    using i512 = integral_constant<int, 512>;
    if(rows <= 256)
        return go(integral_constant<int, 32>{}, integral_constant<int, 1>{}, i256{});
    if(rows <= 512)
        return go(integral_constant<int, 32>{}, integral_constant<int, 1>{}, i512{});
    if(rows <= 1024)
        return go(integral_constant<int, 32>{}, integral_constant<int, 2>{}, i512{});
    if(rows <= 1536)
        return go(integral_constant<int, 32>{}, integral_constant<int, 3>{}, i512{});
    if(rows <= 2048)
        return go(integral_constant<int, 16 * S>{}, integral_constant<int, 4>{}, i512{});
    if(rows <= 4096)
        return go(integral_constant<int, 8 * S>{}, integral_constant<int, 8>{}, i512{});
    if constexpr(sizeof(T) == 4)
        return go(integral_constant<int, 8>{}, integral_constant<int, 16>{}, i512{});
    else
        return rocblas_status_internal_error; // taller than panel_reg_width allows
}

#define RSA_PANEL_INST(T)                                                                       \
    template int panel_reg_width<T>(int, int);                                                  \
    template rocblas_status outer_apply<T>(hipStream_t, int, Batch<T>, int, const int*, int64_t, \
                                           int, int, int, bool, int);                           \
    template rocblas_status panel_reg<T>(hipStream_t, int, Batch<T>, int, int*, int64_t, int*,  \
                                         int, int, int, int, int, int, bool);
RSA_PANEL_INST(float)
RSA_PANEL_INST(double)

} // namespace rsa
