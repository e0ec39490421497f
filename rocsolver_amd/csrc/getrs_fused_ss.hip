// getrs_fused_ss.hip -- instantiates the one-workgroup-per-system solve
// (getrs_fused.hpp) for float.
#include "getrs_fused.hpp"

namespace rsa
{
template <>
rocblas_status getrs_fused<float>(hipStream_t stream, bool trans, int n, int nrhs, Batch<float> A,
                                int lda, const int* ipiv, int64_t strideP, Batch<float> B, int ldb,
                                Batch<float> X, int ldx, int bc, const int* skip)
{
    return getrs_fused_launch<float>(stream, trans, n, nrhs, A, lda, ipiv, strideP, B, ldb, X, ldx, bc,
                                   skip);
}
} // namespace rsa
