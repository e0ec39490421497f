// adjoint.hip -- reverse-mode derivative of the batched solve X = A^-1 B.
//
// Given the LU and pivots of A (getrf/gesv output), the solution X and the
// upstream gradient dX:
//   dB = A^-T dX      -- transposed getrs reusing the stored LU and ipiv
//   dA = -dB X^T      -- batched outer product, this file
// No counterpart in the reference; the transposed solve follows getrs's
// op = T order (roclapack_getrs.hpp:134-150).
#include "internal.hpp"
#include "mfma.hpp"

namespace rsa
{

constexpr int OR = 4; // 16-row tiles of an output column group per wavefront
constexpr int OK = 4; // matrix-core steps (4 right-hand sides each) whose loads are in flight

// dA = -sum_c dB[:, c] X[:, c]^T on the matrix cores: a wavefront forms 64 rows
// of 16 columns, its operands straight from memory (the operands are swapped,
// so that 16 lanes write 16 consecutive rows).  The products accumulate from
// zero as a chain of fused multiply-adds with c increasing.
//
// Bound by writing dA.  No LDS and no barrier, and only the 16-column groups
// and 16-row tiles that hold entries of dA are formed: 64x64 tiles staged in
// LDS with 16 vector fused multiply-adds per staged value took 73 us at n = 96
// x 2048, 16 right-hand sides (151 MB of dA); this kernel takes 49 us.
template <typename T>
__global__ __launch_bounds__(256) void outer_neg_kernel(int n, int nrhs, Batch<T> DB, int lddb,
                                                        Batch<T> XX, int ldx, Batch<T> DA,
                                                        int ldda, int64_t boff)
{
    using M = mfma16<T>;
    const int64_t b = blockIdx.y + boff;
    const int lane = threadIdx.x & 63;
    const unsigned groups = unsigned(n + 15) / 16;
    const unsigned unit = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i0 = int(unit / groups) * 16 * OR;
    const int j0 = int(unit % groups) * 16;
    if(i0 >= n)
        return;
    const int l16 = lane & 15, g = lane >> 4;
    const T* dB = DB[b] + i0 + l16 + int64_t(g) * lddb;
    const T* X = XX[b] + j0 + l16 + int64_t(g) * ldx;
    const int left = n - i0 - l16; // row 16 t + l16 of the wavefront's rows exists: 16 t < left
    const bool xin = j0 + l16 < n;
    typename M::acc_t acc[OR];
#pragma unroll
    for(int t = 0; t < OR; ++t)
        acc[t] = typename M::acc_t{0, 0, 0, 0};
    for(int c0 = 0; c0 < nrhs; c0 += 4 * OK) // uniform
    {
        T xv[OK], bv[OK][OR];
#pragma unroll
        for(int q = 0; q < OK; ++q)
        {
            const int c = c0 + 4 * q;
            const bool in = c + g < nrhs;
            xv[q] = in && xin ? X[int64_t(c) * ldx] : T(0);
#pragma unroll
            for(int t = 0; t < OR; ++t)
                bv[q][t] = in && 16 * t < left ? dB[16 * t + int64_t(c) * lddb] : T(0);
        }
#pragma unroll
        for(int q = 0; q < OK; ++q)
#pragma unroll
            for(int t = 0; t < OR; ++t)
                acc[t] = M::run(xv[q], bv[q][t], acc[t]);
    }
    T* dA = DA[b] + i0 + l16;
#pragma unroll
    for(int r = 0; r < 4; ++r)
    {
        const int j = j0 + M::row(lane, r);
#pragma unroll
        for(int t = 0; t < OR; ++t)
            if(j < n && 16 * t < left)
                dA[16 * t + int64_t(j) * ldda] = -acc[t][r];
    }
}

template <typename T>
__global__ __launch_bounds__(256) void copy_cols_kernel(int n, int ncols, Batch<T> S, int lds,
                                                        Batch<T> D, int ldd, int64_t boff)
{
    const int64_t b = blockIdx.y + boff;
    const T* s = S[b];
    T* d = D[b];
    for(int64_t e = int64_t(blockIdx.x) * 256 + threadIdx.x; e < int64_t(n) * ncols;
        e += int64_t(gridDim.x) * 256)
    {
        const int i = int(e % n), c = int(e / n);
        d[i + int64_t(c) * ldd] = s[i + int64_t(c) * lds];
    }
}

template <typename T>
rocblas_status gesv_adjoint(hipStream_t stream, int n, int nrhs, Batch<T> LU, int lda,
                            const int* ipiv, int64_t strideP, Batch<T> X, int ldx, Batch<T> dX,
                            int lddx, Batch<T> dB, int lddb, Batch<T> dA, int ldda, int bc)
{
    if(n == 0 || bc == 0)
        return rocblas_status_success;
    constexpr int64_t MAXYZ = 65535;
    if(nrhs > 0)
    {
        const bool fused = n <= FUSED_MAX
                           && (n > SMALL_MAX || getrs_small_by_tiles<T>(n, nrhs, bc))
                           && fits_buffer<T>(lda, n)
                           && fits_buffer<T>(lddx, nrhs) && fits_buffer<T>(lddb, nrhs);
        rocblas_status st;
        if(fused) // reads dX, writes dB
            st = getrs_fused<T>(stream, true, n, nrhs, LU, lda, ipiv, strideP, dX, lddx, dB, lddb,
                                bc, nullptr);
        else
        {
            // dB = dX, then dB = A^-T dB
            for(int64_t b0 = 0; b0 < bc; b0 += MAXYZ)
            {
                const int nb = int((bc - b0) < MAXYZ ? (bc - b0) : MAXYZ);
                const int gx = ceil_div(int64_t(n) * nrhs, 256) < 64
                                   ? ceil_div(int64_t(n) * nrhs, 256)
                                   : 64;
                hipLaunchKernelGGL((copy_cols_kernel<T>), dim3(gx, nb), dim3(256), 0, stream, n,
                                   nrhs, dX, lddx, dB, lddb, b0);
                RSA_LAUNCH_CHECK();
            }
            if(n <= SMALL_MAX)
                st = getrs_small<T>(stream, true, n, nrhs, LU, lda, ipiv, strideP, dB, lddb, bc,
                                    true);
            else
                st = getrs_blocked<T>(stream, true, n, nrhs, LU, lda, ipiv, strideP, dB, lddb, bc,
                                      true, nullptr);
        }
        if(st != rocblas_status_success)
            return st;
    }
    // dA = -dB X^T (zero when nrhs == 0)
    for(int64_t b0 = 0; b0 < bc; b0 += MAXYZ)
    {
        const int nb = int((bc - b0) < MAXYZ ? (bc - b0) : MAXYZ);
        // four wavefronts a workgroup, each 16 OR rows of 16 columns
        const int64_t units = int64_t(ceil_div(n, 16)) * ceil_div(n, 16 * OR);
        const dim3 grid(unsigned(ceil_div(units, 4)), nb);
        hipLaunchKernelGGL((outer_neg_kernel<T>), grid, dim3(256), 0, stream, n, nrhs, dB, lddb, X,
                           ldx, dA, ldda, b0);
        RSA_LAUNCH_CHECK();
    }
    return rocblas_status_success;
}

template rocblas_status gesv_adjoint<float>(hipStream_t, int, int, Batch<float>, int, const int*,
                                            int64_t, Batch<float>, int, Batch<float>, int,
                                            Batch<float>, int, Batch<float>, int, int);
template rocblas_status gesv_adjoint<double>(hipStream_t, int, int, Batch<double>, int,
                                             const int*, int64_t, Batch<double>, int,
                                             Batch<double>, int, Batch<double>, int,
                                             Batch<double>, int, int);

} // namespace rsa
