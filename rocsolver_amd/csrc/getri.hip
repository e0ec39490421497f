// getri.hip -- matrix inverse from the LU factorisation (getri,
// getri_outofplace and their no-pivoting variants).
//
// inv(A) is computed as the solution X of A X = I with the triangular-solve
// kernels of the LU path (the row interchanges of ipiv applied to I, then the
// unit-lower and upper solves; up to n = 512 inverse_tile_kernel mostly forms
// the columns of I itself), which is how the reference computes its
// out-of-place inverse (roclapack_getri_outofplace.hpp:100-127).  The in-place
// form (roclapack_getri.hpp:265-378 solves inv(A) L = inv(U) instead) works
// on a copy of the factors in the handle's workspace and writes X over A;
// both forms give the inverse to the reference's test tolerance.  info is the
// first zero on the diagonal of U (1-based, as the reference's trtri /
// check_singularity report it); the inverse is then undefined, as in the
// reference.
#include "internal.hpp"
#include "tile_solve.hpp"

#include <type_traits>

namespace rsa
{

// One wavefront per matrix: the first zero diagonal entry of U.
template <typename T>
__global__ __launch_bounds__(256) void diag_zero_kernel(int n, Batch<T> A, int lda,
                                                        int* __restrict__ info, int bc)
{
    const int64_t b = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if(b >= bc)
        return;
    const int lane = threadIdx.x & 63;
    const T* a = A[b];
    int first = 0;
    for(int i0 = 0; i0 < n; i0 += 64)
    {
        const int i = i0 + lane;
        const bool z = i < n && a[i + int64_t(i) * lda] == T(0);
        const uint64_t m = __builtin_amdgcn_ballot_w64(z);
        if(m != 0) // uniform
        {
            first = i0 + int(__builtin_ctzll(m)) + 1;
            break;
        }
    }
    if(lane == 0)
        info[b] = first;
}

// C = I (n x n, leading dimension ldc) for every batch entry.
template <typename T>
__global__ __launch_bounds__(256) void set_identity_kernel(int n, Batch<T> C, int ldc, int bc)
{
    const int64_t nn = int64_t(n) * n;
    for(int64_t b = blockIdx.y; b < bc; b += gridDim.y)
    {
        T* c = C[b];
        for(int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; e < nn;
            e += int64_t(gridDim.x) * blockDim.x)
        {
            const int i = int(e % n), j = int(e / n);
            c[i + int64_t(j) * ldc] = i == j ? T(1) : T(0);
        }
    }
}

// D = S (n x n) for every batch entry.
template <typename T>
__global__ __launch_bounds__(256) void copy_square_kernel(int n, Batch<T> S, int lds, Batch<T> D,
                                                          int ldd, int bc)
{
    const int64_t nn = int64_t(n) * n;
    for(int64_t b = blockIdx.y; b < bc; b += gridDim.y)
    {
        const T* s = S[b];
        T* d = D[b];
        for(int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; e < nn;
            e += int64_t(gridDim.x) * blockDim.x)
        {
            const int i = int(e % n), j = int(e / n);
            d[i + int64_t(j) * ldd] = s[i + int64_t(j) * lds];
        }
    }
}

static dim3 square_grid(int n, int bc)
{
    const int64_t tiles = (int64_t(n) * n + 255) / 256;
    return dim3(unsigned(tiles < 64 ? tiles : 64), unsigned(bc < 65535 ? bc : 65535));
}

// One system and 16 CT columns of its inverse per workgroup.  Bound by the
// latency of the solves; against writing I and solving for it, the forward
// solve skips the blocks that the identity leaves zero (on average half), and
// no right-hand side is written or read: dgetri n = 100 x 2000 0.81 -> 0.68
// ms with its two copies.  Scratch a lane: 44 bytes in FP64 up to n = 128, 152
// (FP32 36) up to 256, 12 (36) beyond; with SUMS 28 (36) and 20 (28).
//
// SUMS (no interchanges, n > 64): a row adds sums of 32 products, not a chain of
// n; with interchanges every column has the bits of a solve for it.  FP32 errors
// against 64 bits, chain -> sums: n = 512, random 5.8e-6 -> 3.9e-6, diagonally
// dominant 4.3e-7 -> 1.4e-7; n = 200 1.9e-6 -> 1.6e-6, 2.7e-7 -> 1.3e-7.  Times
// with the chain and with sums: n = 200 x 2000 FP32 0.96 and 0.98 ms, FP64 2.22
// and 1.84; n = 400 x 512 FP64 2.82 and 2.86.
template <typename T, int NMAX, int NT, int CT, bool SUMS>
__global__ __launch_bounds__(NT, (tile_waves<T, NMAX, NT>())) void inverse_tile_kernel(
    int n, Batch<T> AA, int lda, const int* __restrict__ ipivA, int64_t strideP, Batch<T> XX,
    int ldx, int bc, unsigned chunks)
{
    unsigned chunk;
    const int64_t b = tile_solve_system(blockIdx.x, chunks, chunk);
    if(b >= bc)
        return;
    tile_inverse_body<T, NMAX, NT, CT, SUMS>(n, int(chunk) * CT * TSC, AA[b], lda,
                                   ipivA ? ipivA + b * strideP : nullptr, XX[b], ldx);
}

// Tiles against the team solve of lu_small.hpp (eight columns of the inverse a
// pass, several systems per wavefront), which is the faster one for small
// orders in large batches.  Team against tiles, FP64: n = 64 x 8192 1.80
// against 0.66 ms, n = 32 x 8192 248 against 183 us, n = 24 x 8192 148 against
// 173 but x 1024 63 against 39, n = 16 x 1024 31 against 19.
inline bool inverse_by_tiles(int n, int bc)
{
    return n > 24 || (n > 8 && bc <= 1024);
}

template <typename T>
static rocblas_status inverse_tiles(hipStream_t stream, int n, Batch<T> LU, int ldlu,
                                    const int* ipiv, int64_t strideP, Batch<T> X, int ldx, int bc)
{
    using std::integral_constant;
    // 32 columns a workgroup beyond n = 128: n = 400 x 200 2.02 -> 1.35 ms, n =
    // 200 x 800 1.31 -> 1.13; no gain at n = 100 (0.68), 0.96 at n = 128 x 100
    const int cols = n <= 128 ? TSC : 2 * TSC;
    const int chunks = ceil_div(n, cols); // at most 16: never split
    auto go = [&](auto nmax, auto nt, auto ct) {
        constexpr int NMAX = decltype(nmax)::value;
        constexpr int NT = decltype(nt)::value;
        constexpr int CT = decltype(ct)::value;
        auto* kernel = inverse_tile_kernel<T, NMAX, NT, CT, false>;
        if constexpr(NMAX > 64)
            if(!ipiv)
                kernel = inverse_tile_kernel<T, NMAX, NT, CT, true>;
        return launch_split(
            bc, chunks, NT, TILE_XCDS, [&](int64_t b0, int64_t nb, int64_t, int64_t) {
                hipLaunchKernelGGL(kernel,
                                   dim3(unsigned(tile_solve_grid(int(nb), chunks))), dim3(NT), 0,
                                   stream, n, batch_from(LU, b0), ldlu,
                                   ipiv ? ipiv + b0 * strideP : nullptr, strideP,
                                   batch_from(X, b0), ldx, int(nb), unsigned(chunks));
                RSA_LAUNCH_CHECK();
                return rocblas_status_success;
            });
    };
    constexpr int F = sizeof(T) == 8 ? 2 : 1; // as getrs_fused_launch
    if(n <= 64)
        return go(integral_constant<int, 64>{}, integral_constant<int, 64 * F>{},
                  integral_constant<int, 1>{});
    if(n <= 128)
        return go(integral_constant<int, 128>{}, integral_constant<int, 128 * F>{},
                  integral_constant<int, 1>{});
    if(n <= 256)
        return go(integral_constant<int, 256>{}, integral_constant<int, 256 * F>{},
                  integral_constant<int, 2>{});
    return go(integral_constant<int, 512>{}, integral_constant<int, 512>{},
              integral_constant<int, 2>{});
}

template <typename T>
rocblas_status getri_solve(hipStream_t stream, int n, Batch<T> LU, int ldlu, const int* ipiv,
                           int64_t strideP, Batch<T> X, int ldx, int* info, int bc, bool pivot)
{
    if(n <= 0 || bc <= 0)
        return rocblas_status_success;
    const rocblas_status st
        = launch_split(bc, 1, 64, 4, [&](int64_t b0, int64_t nb, int64_t, int64_t) {
              hipLaunchKernelGGL((diag_zero_kernel<T>), dim3(ceil_div(nb, 4)), dim3(256), 0, stream,
                                 n, batch_from(LU, b0), ldlu, info + b0, int(nb));
              RSA_LAUNCH_CHECK();
              return rocblas_status_success;
          });
    if(st != rocblas_status_success)
        return st;
    if(inverse_by_tiles(n, bc) && n <= FUSED_MAX && fits_buffer<T>(ldlu, n) && fits_buffer<T>(ldx, n))
        return inverse_tiles<T>(stream, n, LU, ldlu, pivot ? ipiv : nullptr, strideP, X, ldx, bc);
    hipLaunchKernelGGL((set_identity_kernel<T>), square_grid(n, bc), dim3(256), 0, stream, n, X,
                       ldx, bc);
    RSA_LAUNCH_CHECK();
    if(n <= SMALL_MAX)
        return getrs_small<T>(stream, false, n, n, LU, ldlu, ipiv, strideP, X, ldx, bc, pivot);
    return getrs_blocked<T>(stream, false, n, n, LU, ldlu, ipiv, strideP, X, ldx, bc, pivot,
                            nullptr);
}

template <typename T>
rocblas_status copy_square(hipStream_t stream, int n, Batch<T> S, int lds, Batch<T> D, int ldd,
                           int bc)
{
    if(n <= 0 || bc <= 0)
        return rocblas_status_success;
    hipLaunchKernelGGL((copy_square_kernel<T>), square_grid(n, bc), dim3(256), 0, stream, n, S,
                       lds, D, ldd, bc);
    RSA_LAUNCH_CHECK();
    return rocblas_status_success;
}

#define RSA_GETRI_INST(T)                                                                     \
    template rocblas_status getri_solve<T>(hipStream_t, int, Batch<T>, int, const int*,       \
                                           int64_t, Batch<T>, int, int*, int, bool);          \
    template rocblas_status copy_square<T>(hipStream_t, int, Batch<T>, int, Batch<T>, int, int);
RSA_GETRI_INST(float)
RSA_GETRI_INST(double)

} // namespace rsa
