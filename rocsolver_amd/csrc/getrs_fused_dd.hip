// getrs_fused_dd.hip -- instantiates the one-workgroup-per-system solve
// (getrs_fused.hpp) for double.
#include "getrs_fused.hpp"

namespace rsa
{
template <>
rocblas_status getrs_fused<double>(hipStream_t stream, bool trans, int n, int nrhs, Batch<double> A,
                                int lda, const int* ipiv, int64_t strideP, Batch<double> B, int ldb,
                                Batch<double> X, int ldx, int bc, const int* skip)
{
    return getrs_fused_launch<double>(stream, trans, n, nrhs, A, lda, ipiv, strideP, B, ldb, X, ldx, bc,
                                   skip);
}
} // namespace rsa
