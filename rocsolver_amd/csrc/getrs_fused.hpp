// getrs_fused.hpp -- one-workgroup-per-system triangular solves with the LU
// of getrf, for n <= FUSED_MAX (reference order of operations:
// library/src/lapack/roclapack_getrs.hpp:117-150 -- laswp, then L, then U for
// op = N; U^T, L^T, then the reverse interchanges for op = T).  The factors
// are read through a buffer resource: lda * n * sizeof(T) must be below 2^31
// (fits_buffer).  Systems with skip[b] != 0 are left untouched.
//
// Two kernels with the same operations per row, so bit-identical results:
//   * the tile solver of tile_solve.hpp, 16 right-hand sides per workgroup;
//   * beyond n = 64, the row solver of trsv_rows.hpp, thread i owning row i of
//     up to eight right-hand sides, for large batches with few of them
//     (rows_rule.hpp).
#pragma once

#include "rows_rule.hpp"
#include "tile_solve.hpp"
#include "trsv_rows.hpp"

#include <type_traits>

namespace rsa
{

template <typename T, int NMAX, int NT, bool TRANS>
__global__ __launch_bounds__(NT, (tile_waves<T, NMAX, NT>())) void getrs_tile_kernel(
    int n, int nrhs, Batch<T> AA, int lda, const int* __restrict__ ipivA, int64_t strideP,
    Batch<T> BB, int ldb, Batch<T> XX, int ldx, int bc, unsigned chunks, unsigned chunk0,
    const int* __restrict__ skip)
{
    unsigned chunk;
    const int64_t b = tile_solve_system(blockIdx.x, chunks, chunk);
    if(b >= bc || (skip && skip[b] != 0))
        return;
    const int c0 = int(chunk0 + chunk) * TSC;
    const int cend = nrhs - c0 < TSC ? nrhs : c0 + TSC;
    tile_solve_body<T, NMAX, NT, TILE_LU, TRANS>(n, c0, cend, AA[b], lda, ipivA + b * strideP,
                                                 BB[b], ldb, XX[b], ldx);
}

// One system per workgroup (blockDim.x == NMAX, n <= NMAX), nrhs <= NR.
template <typename T, int NMAX, int NR, bool TRANS>
__global__ __launch_bounds__(NMAX) void getrs_rows_kernel(int n, int nrhs, Batch<T> AA, int lda,
                                                          const int* __restrict__ ipivA,
                                                          int64_t strideP, Batch<T> BB, int ldb,
                                                          Batch<T> XX, int ldx,
                                                          const int* __restrict__ skip)
{
    __shared__ T sx[2][GBS][NR];
    __shared__ T sL[GBS][GBS + 1];
    __shared__ int sipiv[NMAX];
    __shared__ int ssrc[NMAX];

    const int64_t b = blockIdx.x;
    if(skip && skip[b] != 0)
        return;
    const int tid = threadIdx.x;
    const MatrixBuffer<T> A(AA[b], lda, n);
    const MatrixBuffer<T> Bbuf(BB[b], ldb, nrhs);
    T* X = XX[b];
    const int pos = pivot_position(n, ipivA + b * strideP, TRANS, sipiv, ssrc);
    const int src = TRANS ? tid : ssrc[tid];
    const int dst = TRANS ? pos : tid;

    // all loads issued back to back (out-of-range offsets read 0)
    T x[NR];
#pragma unroll
    for(int q = 0; q < NR; ++q)
    {
        const uint32_t off = (tid < n && q < nrhs) ? Bbuf.row_offset(src) + Bbuf.col_offset(q)
                                                   : MatrixBuffer<T>::OUT_OF_RANGE;
        x[q] = Bbuf.load(off, 0);
    }
    solve_lower_rows<T, NR, TRANS>(n, A, x, sx, sL);
    solve_upper_rows<T, NR, TRANS>(n, A, x, sx, sL);
    // every thread has read its right-hand side before any row is stored
    // (X may alias B and op = T stores at the permuted row)
    __syncthreads();
    if(tid < n)
    {
#pragma unroll
        for(int q = 0; q < NR; ++q)
            if(q < nrhs)
                X[dst + int64_t(q) * ldx] = x[q];
    }
}

template <typename T>
rocblas_status getrs_fused_launch(hipStream_t stream, bool trans, int n, int nrhs, Batch<T> A,
                                  int lda, const int* ipiv, int64_t strideP, Batch<T> B, int ldb,
                                  Batch<T> X, int ldx, int bc, const int* skip)
{
    using std::integral_constant;
    if(bc <= 0 || n <= 0 || nrhs <= 0)
        return rocblas_status_success;
    if(n > SMALL_MAX && getrs_by_rows<T>(trans, n, nrhs, bc))
    {
        auto go = [&](auto nmax, auto nr, auto tr) {
            constexpr int NMAX = decltype(nmax)::value;
            constexpr int NR = decltype(nr)::value;
            constexpr bool TR = decltype(tr)::value;
            return launch_split(bc, 1, NMAX, 1, [&](int64_t b0, int64_t nb, int64_t, int64_t) {
                hipLaunchKernelGGL((getrs_rows_kernel<T, NMAX, NR, TR>), dim3(unsigned(nb)),
                                   dim3(NMAX), 0, stream, n, nrhs, batch_from(A, b0), lda,
                                   ipiv + b0 * strideP, strideP, batch_from(B, b0), ldb,
                                   batch_from(X, b0), ldx, skip ? skip + b0 : nullptr);
                RSA_LAUNCH_CHECK();
                return rocblas_status_success;
            });
        };
        auto by_nrhs = [&](auto nmax, auto tr) {
            return nrhs == 1 ? go(nmax, integral_constant<int, 1>{}, tr)
                             : go(nmax, integral_constant<int, 4>{}, tr);
        };
        // the orders and right-hand sides that getrs_by_rows can give
        if(n <= 128)
            return trans ? by_nrhs(integral_constant<int, 128>{}, std::true_type{})
                         : by_nrhs(integral_constant<int, 128>{}, std::false_type{});
        if(n <= 256)
            return trans ? by_nrhs(integral_constant<int, 256>{}, std::true_type{})
                         : by_nrhs(integral_constant<int, 256>{}, std::false_type{});
        if(nrhs > 4)
            return go(integral_constant<int, 512>{}, integral_constant<int, 8>{},
                      std::false_type{});
        return by_nrhs(integral_constant<int, 512>{}, std::false_type{});
    }
    auto go = [&](auto nmax, auto nt) {
        constexpr int NMAX = decltype(nmax)::value;
        constexpr int NT = decltype(nt)::value;
        return launch_split(
            bc, ceil_div(nrhs, TSC), NT, TILE_XCDS,
            [&](int64_t b0, int64_t nb, int64_t c0, int64_t nc) {
                const dim3 grid{unsigned(tile_solve_grid(int(nb), int(nc)))};
                const int* sk = skip ? skip + b0 : nullptr;
                if(trans)
                    hipLaunchKernelGGL((getrs_tile_kernel<T, NMAX, NT, true>), grid, dim3(NT), 0,
                                       stream, n, nrhs, batch_from(A, b0), lda,
                                       ipiv + b0 * strideP, strideP, batch_from(B, b0), ldb,
                                       batch_from(X, b0), ldx, int(nb), unsigned(nc), unsigned(c0),
                                       sk);
                else
                    hipLaunchKernelGGL((getrs_tile_kernel<T, NMAX, NT, false>), grid, dim3(NT), 0,
                                       stream, n, nrhs, batch_from(A, b0), lda,
                                       ipiv + b0 * strideP, strideP, batch_from(B, b0), ldb,
                                       batch_from(X, b0), ldx, int(nb), unsigned(nc), unsigned(c0),
                                       sk);
                RSA_LAUNCH_CHECK();
                return rocblas_status_success;
            });
    };
    // FP64: two tiles a wavefront up to n = 256 (n = 96 x 2048 78 us
    // against 91 with four, n = 256 x 4096 681 against 713); FP32: four
    // (49 against 58 us, 367 against 493)
    constexpr int F = sizeof(T) == 8 ? 2 : 1;
    if(n <= 64)
        return go(integral_constant<int, 64>{}, integral_constant<int, 64 * F>{});
    if(n <= 128)
        return go(integral_constant<int, 128>{}, integral_constant<int, 128 * F>{});
    if(n <= 256)
        return go(integral_constant<int, 256>{}, integral_constant<int, 256 * F>{});
    return go(integral_constant<int, 512>{}, integral_constant<int, 512>{});
}

} // namespace rsa
