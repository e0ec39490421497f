// tile_solve.hpp -- triangular solves of one system per workgroup on the
// matrix cores, up to 16 right-hand sides at a time.
//
// The right-hand sides live in MFMA accumulators, 16 rows x 16 columns per
// tile, tile t on wavefront t % NW (a column of the triangle shrinks or grows
// over all of them evenly).  Each triangle is walked in 32-row diagonal
// blocks (two barriers per block):
//   * the wavefronts holding the block's rows subtract the previous block's
//     columns from them and publish them to LDS, all threads the 32x32
//     diagonal block, loaded one block ahead;
//   * one wavefront solves the block, four lanes per right-hand side
//     (quad_solve.hpp), while the others subtract the previous block's
//     columns from the tiles beyond: eight v_mfma_*_16x16x4 a tile, their
//     entries of op(A) read straight from memory one block ahead.
// v_mfma_*_16x16x4 adds its four products as a chain of fused multiply-adds
// with k increasing (checked bit for bit on gfx950, FP32 and FP64), so with
// accumulators that start at B, the solution negated, and for a backward
// solve the four k in reverse, every row is updated in the column order of
// the reference's substitution, one fused multiply-add per entry
// (library/src/lapack/roclapack_getrs.hpp:117-150); the diagonal is applied
// by true division.
//
// Bound by latency per system (n / 32 steps per triangle) and by reading the
// factor.  Measured (FP64, 16 right-hand sides, against a row per thread with
// vector fused multiply-adds and eight right-hand sides a pass): n = 96 x 2048
// 202 -> 78 us, transposed 287 -> 84; n = 256 x 4096 1355 -> 681 us,
// transposed 2072 -> 800; one n = 128 system 127 -> 34 us.
#pragma once

#include "internal.hpp"
#include "mfma.hpp"
#include "quad_solve.hpp"

namespace rsa
{

constexpr int TSB = 32; // diagonal block
constexpr int TSC = 16; // right-hand sides per pass
constexpr int TSX = TSB + 1; // column stride of the block's right-hand sides in LDS

// tiles per wavefront: rows of a system on NT threads, n <= NMAX
template <int NMAX, int NT>
constexpr int tile_solve_tpw()
{
    return NMAX / 16 / (NT / 64);
}

// Wavefronts per SIMD that the registers are cut for: two tiles a wavefront
// fit four, four tiles two in FP64.  (At NMAX = 64 the LDS holds six workgroups
// of two wavefronts a CU, three a SIMD.)  At four the FP64 kernels of n <= 256
// keep 12 to 52 bytes a lane in scratch; four tiles a wavefront, two a SIMD,
// took 91 us for 78 at n = 96 x 2048.
template <typename T, int NMAX, int NT>
constexpr int tile_waves()
{
    return sizeof(T) == 4 ? 4 : NMAX == 64 ? 3 : NMAX < NT ? 4 : 2;
}

// op(T) X = acc in place, T the lower (forward) or upper (backward) triangle
// of op(A).  Rows past n are zero in and out.  par: parity of the LDS buffers.
// A forward solve starts at block `begin` (the rows before it are zero).  CT
// groups of 16 right-hand sides share the factor's entries and the barriers;
// each has its own solving wavefront.  SUMS: a block's 32 products are summed
// from zero before they are added to a row, so that a row's chain is n / 32
// sums long in place of n products.
template <typename T, int NT, int TPW, int CT, bool LOWER, bool TRANS, bool UNIT,
          bool SUMS = false>
__device__ __forceinline__ void tile_solve_triangle(int n, const MatrixBuffer<T>& A,
                                                    typename mfma16<T>::acc_t (&acc)[TPW][CT],
                                                    T (*sX)[CT * TSC * TSX],
                                                    T (*sL)[TSB * TSB],
                                                    int& par, int begin = 0)
{
    using M = mfma16<T>;
    constexpr int NW = NT / 64;
    static_assert(CT <= NW, "a solving wavefront per group");
    constexpr int DL = TSB * TSB / NT; // entries of the diagonal block per thread
    constexpr int KS = TSB / 4;
    // Solved values read where they are used, not ahead: the sums leave no
    // registers for them at n = 129 to 256 in FP64 (204 -> 28 bytes of scratch a
    // lane, n = 200 x 2000 2.50 -> 1.84 ms; up to 512, with none to spare in
    // either, 5 % slower)
    constexpr bool LATE = SUMS && sizeof(T) == 8 && CT > 1 && TPW == 2;
    const int D = (n + TSB - 1) / TSB;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    T av[TPW][KS], dl[DL];
    auto load_diag = [&](int d) {
        const int ft = fresh_tid();
#pragma unroll
        for(int h = 0; h < DL; ++h)
        {
            const int e = ft + h * NT, x = TSB * d + e % TSB, y = TSB * d + e / TSB;
            dl[h] = A.load(A.offset(x < n && y < n, x, y), 0);
        }
    };
    auto put_diag = [&](int d, T* L) { // past n: the identity
        const int ft = fresh_tid();
#pragma unroll
        for(int h = 0; h < DL; ++h)
        {
            const int e = ft + h * NT, x = e % TSB, y = e / TSB;
            const bool in = TSB * d + x < n && TSB * d + y < n;
            L[TRANS ? x * TSB + y : e] = in ? dl[h] : (x == y ? T(1) : T(0));
        }
    };
    auto beyond = [&](int tile, int d) { // uniform
        return (LOWER ? tile > 2 * d + 1 : tile < 2 * d) && 16 * tile < n;
    };
    auto load_rows = [&](int d) { // this wavefront's rows beyond block d
        const int lane = fresh_tid() & 63;
        const int g = LOWER ? lane >> 4 : 3 - (lane >> 4);
#pragma unroll
        for(int t = 0; t < TPW; ++t)
        {
            const int tile = wid + t * NW; // uniform
            // an inactive tile or a row past n reads nothing
            const bool act = beyond(tile, d) && 16 * tile + (lane & 15) < n;
#pragma unroll
            for(int ks = 0; ks < KS; ++ks)
            {
                const int k = TSB * d + 4 * ks; // + g
                const bool in = act && k + g < n;
                if constexpr(TRANS)
                    av[t][ks] = A.load(in ? A.col_offset(lane & 15) + A.row_offset(g)
                                          : MatrixBuffer<T>::OUT_OF_RANGE,
                                       A.col_offset(16 * tile) + A.row_offset(k));
                else
                    av[t][ks] = A.load(in ? A.row_offset(lane & 15) + A.col_offset(g)
                                          : MatrixBuffer<T>::OUT_OF_RANGE,
                                       A.row_offset(16 * tile) + A.col_offset(k));
            }
        }
    };
    auto publish = [&](int t, int tile, T* X) {
        const int lane = fresh_tid() & 63;
#pragma unroll
        for(int ct = 0; ct < CT; ++ct)
#pragma unroll
            for(int r = 0; r < 4; ++r)
                X[(16 * ct + M::row(lane, r)) * TSX + 16 * (tile & 1) + (lane & 15)]
                    = acc[t][ct][r];
    };
    auto solve = [&](int ct, int d, T* X, const T* L) { // group ct, by one wavefront
        const int lane = fresh_tid() & 63;
        T x[TSB / 4];
        T* xp = X + (16 * ct + (lane >> 2)) * TSX + (lane & 3);
#pragma unroll
        for(int q = 0; q < TSB / 4; ++q)
            x[q] = xp[4 * q];
        // fewer columns ahead where registers bound the resident wavefronts
        constexpr int G = sizeof(T) == 8 && TPW > 2 ? 2 : sizeof(T) == 8 ? 1 : 2;
        quad_solve<T, TSB, LOWER, UNIT, G>(L, lane, x);
#pragma unroll
        for(int q = 0; q < TSB / 4; ++q)
            // rows past n stay zero (an infinite solution times the padding's
            // zeros is not)
            xp[4 * q] = TSB * d + 4 * q + (lane & 3) < n ? x[q] : T(0);
    };

    const int first = LOWER ? begin : D - 1, dir = LOWER ? 1 : -1;
    const int steps = D - begin;
    load_diag(first);
#pragma unroll
    for(int t = 0; t < TPW; ++t)
        if(((wid + t * NW) >> 1) == first) // uniform
            publish(t, wid + t * NW, sX[par]);
    put_diag(first, sL[par]);
    load_rows(first);
    if(steps > 1) // uniform
        load_diag(first + dir);
    __syncthreads();
    if(wid < CT)
        solve(wid, first, sX[par], sL[par]);
    __syncthreads();
    for(int s = 0; s < steps; ++s)
    {
        // block d is solved; its product with the rows of the next block
        // comes first, so that the next block is solved while the other
        // wavefronts update the rows beyond it
        const int d = first + dir * s, next = d + dir;
        const bool more = s + 1 < steps; // uniform
        T* X = sX[par];
        T* Xn = sX[par ^ 1];
        T* Ln = sL[par ^ 1];
        par ^= 1;
        T bv[CT][KS];
        auto load_solved = [&](int ct) {
            const int lane = fresh_tid() & 63;
            const int g = LOWER ? lane >> 4 : 3 - (lane >> 4);
#pragma unroll
            for(int ks = 0; ks < KS; ++ks)
                bv[ct][ks] = -X[(16 * ct + (lane & 15)) * TSX + 4 * ks + g];
        };
        if constexpr(!LATE)
#pragma unroll
            for(int ct = 0; ct < CT; ++ct)
                load_solved(ct);
        auto update = [&](int t) {
            if constexpr(SUMS)
            {
#pragma unroll
                for(int ct = 0; ct < CT; ++ct)
                {
                    if constexpr(LATE)
                        load_solved(ct);
                    typename M::acc_t sum = {0, 0, 0, 0};
#pragma unroll
                    for(int q = 0; q < KS; ++q)
                    {
                        const int ks = LOWER ? q : KS - 1 - q;
                        sum = M::run(bv[ct][ks], av[t][ks], sum);
                    }
#pragma unroll
                    for(int r = 0; r < 4; ++r)
                        acc[t][ct][r] += sum[r];
                }
                return;
            }
#pragma unroll
            for(int q = 0; q < KS; ++q)
            {
                const int ks = LOWER ? q : KS - 1 - q;
#pragma unroll
                for(int ct = 0; ct < CT; ++ct)
                    acc[t][ct] = M::run(bv[ct][ks], av[t][ks], acc[t][ct]);
            }
        };
#pragma unroll
        for(int t = 0; t < TPW; ++t)
        {
            const int tile = wid + t * NW;
            if((tile >> 1) == d) // uniform
            {
                const int lane = fresh_tid() & 63;
#pragma unroll
                for(int ct = 0; ct < CT; ++ct)
#pragma unroll
                    for(int r = 0; r < 4; ++r)
                        acc[t][ct][r]
                            = X[(16 * ct + M::row(lane, r)) * TSX + 16 * (tile & 1) + (lane & 15)];
            }
            else if(more && (tile >> 1) == next) // uniform
            {
                if(beyond(tile, d))
                    update(t);
                publish(t, tile, Xn);
            }
        }
        if(!more)
            break;
        put_diag(next, Ln);
        __syncthreads();
        const int ct = (wid + NW - (2 * next) % NW) % NW; // uniform
        if(ct < CT) // first the owners of the next block's rows
            solve(ct, next, Xn, Ln);
#pragma unroll
        for(int t = 0; t < TPW; ++t)
        {
            const int tile = wid + t * NW;
            if((tile >> 1) != next && beyond(tile, d)) // uniform
                update(t);
        }
        load_rows(next);
        if(s + 2 < steps) // uniform
            load_diag(next + dir);
        __syncthreads();
    }
}

// Interchanges of ipiv (1-based, LAPACK order; a pivot outside [1, n] is
// ignored) as a table: row i of P B is row s_row[i] of B, n <= NMAX.  Blocks
// of 64 interchanges are composed by one wavefront each, then applied in
// order by the first.  s_tmp: 3 * NMAX entries.  Ends with a barrier.
template <int NMAX, int NT>
__device__ __forceinline__ void pivot_rows(int n, const int* __restrict__ ipiv,
                                           unsigned short* s_row, unsigned short* s_tmp)
{
    static_assert(NMAX % 64 == 0, "whole blocks");
    const int tid = fresh_tid();
    const int lane = tid & 63;
    const int nblk = (n + 63) / 64;
    unsigned short* s_pos = s_tmp;
    unsigned short* s_src0 = s_tmp + NMAX;
    unsigned short* s_src1 = s_tmp + 2 * NMAX;
    for(int i = tid; i < NMAX; i += NT)
        s_row[i] = (unsigned short)i;
    for(int blk = tid >> 6; blk < nblk; blk += NT / 64)
    {
        const int base = 64 * blk, i = base + lane;
        int p = i < n ? ipiv[i] - 1 : i;
        p = (p >= 0 && p < n) ? p : i;
        int s0 = i, s1 = p;
#pragma unroll 8
        for(int k = 63; k >= 0; --k) // back through the block's interchanges
        {
            const int row = base + k;
            const int q = __builtin_amdgcn_readlane(p, k);
            s0 = s0 == row ? q : (s0 == q ? row : s0);
            s1 = s1 == row ? q : (s1 == q ? row : s1);
        }
        // a partner inside the block is one of its rows; one met twice is
        // moved twice, the same row to the same place
        const bool inside = p >= base && p < base + 64;
        s_src0[i] = (unsigned short)s0;
        s_pos[i] = (unsigned short)(inside ? i : p);
        s_src1[i] = (unsigned short)(inside ? s0 : s1);
    }
    __syncthreads();
    if(tid < 64)
        for(int blk = 0; blk < nblk; ++blk)
        {
            const int i = 64 * blk + lane;
            const int pos = s_pos[i];
            const unsigned short r0 = s_row[s_src0[i]], r1 = s_row[s_src1[i]];
            wave_sync();
            s_row[i] = r0;
            s_row[pos] = r1;
            wave_sync();
        }
    __syncthreads();
}

enum TileFactor : int
{
    TILE_LU = 0, // P A = L U: L unit lower, U upper, rows by ipiv
    TILE_CHOL_L = 1, // A = L L^T, lower storage
    TILE_CHOL_U = 2 // A = U^T U, upper storage
};

// Solves one system with the whole workgroup (blockDim.x == NT, n <= NMAX):
// right-hand sides c0 .. cend-1 of B, 16 at a time, into X (which may be B).
template <typename T, int NMAX, int NT, int FACTOR, bool TRANS>
__device__ __forceinline__ void tile_solve_body(int n, int c0, int cend, const T* __restrict__ Ap,
                                                int lda, const int* __restrict__ ipiv,
                                                const T* Bm, int ldb, T* Xm, int ldx)
{
    using M = mfma16<T>;
    constexpr int NW = NT / 64;
    constexpr int TPW = tile_solve_tpw<NMAX, NT>();
    static_assert(TPW >= 1 && TPW * 16 * NW == NMAX, "whole tiles");
    __shared__ T sX[2][TSC * TSX];
    __shared__ __align__(16) T sL[2][TSB * TSB];
    __shared__ unsigned short s_row[FACTOR == TILE_LU ? NMAX : 1];

    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const MatrixBuffer<T> A(Ap, lda, n);
    const MatrixBuffer<T> B(Bm, ldb, cend), X(Xm, ldx, cend);
    if constexpr(FACTOR == TILE_LU)
    {
        static_assert(sizeof(T) * 2 * TSB * TSB >= 2 * 3 * NMAX, "scratch in sL");
        pivot_rows<NMAX, NT>(n, ipiv, s_row, reinterpret_cast<unsigned short*>(sL));
    }
    // accumulator register r of tile t: row 16 tile + lane % 16, column
    // M::row(lane, r)
    auto offset = [&](const MatrixBuffer<T>& V, int t, int r, bool permuted) {
        const int lane = fresh_tid() & 63;
        const int i = 16 * (wid + t * NW) + (lane & 15);
        const int c = c0 + M::row(lane, r);
        int row = i;
        if constexpr(FACTOR == TILE_LU)
            if(permuted && i < n)
                row = s_row[i];
        return V.offset(i < n && c < cend, row, c);
    };
    int par = 0;
    for(; c0 < cend; c0 += TSC) // uniform
    {
        typename M::acc_t acc[TPW][1];
#pragma unroll
        for(int t = 0; t < TPW; ++t)
#pragma unroll
            for(int r = 0; r < 4; ++r)
                acc[t][0][r] = B.load(offset(B, t, r, !TRANS), 0);
        if constexpr(FACTOR == TILE_LU && !TRANS)
        {
            tile_solve_triangle<T, NT, TPW, 1, true, false, true>(n, A, acc, sX, sL, par);
            tile_solve_triangle<T, NT, TPW, 1, false, false, false>(n, A, acc, sX, sL, par);
        }
        else if constexpr(FACTOR == TILE_LU)
        {
            tile_solve_triangle<T, NT, TPW, 1, true, true, false>(n, A, acc, sX, sL, par); // U^T
            tile_solve_triangle<T, NT, TPW, 1, false, true, true>(n, A, acc, sX, sL, par); // L^T
        }
        else
        {
            constexpr bool UP = FACTOR == TILE_CHOL_U;
            tile_solve_triangle<T, NT, TPW, 1, true, UP, false>(n, A, acc, sX, sL, par);
            tile_solve_triangle<T, NT, TPW, 1, false, !UP, false>(n, A, acc, sX, sL, par);
        }
        // every right-hand side was read before the solves' barriers, so the
        // permuted rows of op T may overwrite them
#pragma unroll
        for(int t = 0; t < TPW; ++t)
#pragma unroll
            for(int r = 0; r < 4; ++r)
                X.store(acc[t][0][r], offset(X, t, r, TRANS), 0);
    }
}

// Columns c0 .. c0 + 16 CT - 1 of U^-1 L^-1 into X, the inverse of A = P^T L U with its
// columns in the order of the interchanges: X = (U^-1 L^-1) P, so column k of
// the product is column s_row[k] of X (ipiv null: no interchanges).  The
// right-hand sides are columns of the identity, formed here; their rows before
// block c0 / 32 are zero through the forward solve, which starts there.
template <typename T, int NMAX, int NT, int CT, bool SUMS>
__device__ __forceinline__ void tile_inverse_body(int n, int c0, const T* __restrict__ Ap, int lda,
                                                  const int* __restrict__ ipiv, T* Xm, int ldx)
{
    using M = mfma16<T>;
    constexpr int NW = NT / 64;
    constexpr int TPW = tile_solve_tpw<NMAX, NT>();
    __shared__ T sX[2][CT * TSC * TSX];
    __shared__ __align__(16) T sL[2][TSB * TSB];
    __shared__ unsigned short s_row[NMAX];

    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const MatrixBuffer<T> A(Ap, lda, n), X(Xm, ldx, n);
    if(ipiv) // uniform
        pivot_rows<NMAX, NT>(n, ipiv, s_row, reinterpret_cast<unsigned short*>(sL));
    else
    {
        for(int i = threadIdx.x; i < NMAX; i += NT)
            s_row[i] = (unsigned short)i;
        __syncthreads();
    }
    typename M::acc_t acc[TPW][CT];
#pragma unroll
    for(int t = 0; t < TPW; ++t)
#pragma unroll
        for(int r = 0; r < 4 * CT; ++r)
        {
            const int lane = fresh_tid() & 63;
            const int i = 16 * (wid + t * NW) + (lane & 15);
            const int k = c0 + 16 * (r / 4) + M::row(lane, r % 4);
            acc[t][r / 4][r % 4] = i < n && i == k ? T(1) : T(0);
        }
    int par = 0;
    tile_solve_triangle<T, NT, TPW, CT, true, false, true, SUMS>(n, A, acc, sX, sL, par, c0 / TSB);
    tile_solve_triangle<T, NT, TPW, CT, false, false, false, SUMS>(n, A, acc, sX, sL, par);
#pragma unroll
    for(int t = 0; t < TPW; ++t)
#pragma unroll
        for(int r = 0; r < 4 * CT; ++r)
        {
            const int lane = fresh_tid() & 63;
            const int i = 16 * (wid + t * NW) + (lane & 15);
            const int k = c0 + 16 * (r / 4) + M::row(lane, r % 4);
            const bool in = i < n && k < n;
            X.store(acc[t][r / 4][r % 4], X.offset(in, i, in ? int(s_row[k]) : 0), 0);
        }
}

// System and group of 16 right-hand sides of a workgroup.  Workgroups go
// round-robin to the 8 XCDs in launch order: the groups of one system are
// given to one XCD, so that its factor is read into one L2.
constexpr int TILE_XCDS = 8;
__device__ __forceinline__ int64_t tile_solve_system(unsigned id, unsigned chunks, unsigned& chunk)
{
    chunk = (id / TILE_XCDS) % chunks;
    return int64_t(id / (TILE_XCDS * chunks)) * TILE_XCDS + id % TILE_XCDS;
}
inline int64_t tile_solve_grid(int bc, int chunks)
{
    return int64_t(ceil_div(bc, TILE_XCDS)) * TILE_XCDS * chunks;
}

} // namespace rsa
