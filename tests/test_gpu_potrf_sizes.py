"""potrf at the edges of its dispatch: the factor is the oracle's bit for bit.

Workgroups of 1, 2 and 4 wavefronts (n <= 64, <= 128, larger); block columns of 32 with
partial last ones; more rows than one pass of the wavefronts covers (128 rows per pass of the
largest workgroup).
"""
import numpy as np
import pytest

import oracle
import rocsolver_amd as ra

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 16, 17, 31, 33, 64, 65, 95, 128, 129, 160, 161, 289, 530])
@pytest.mark.parametrize("uplo", ["L", "U"])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_potrf_bits(torch_gpu, handle, n, uplo, dtype):
    print(f"potrf n={n} {uplo} {dtype.__name__}", flush=True)
    g = np.random.default_rng(n)
    bc, lda = 3, n + 2
    A0 = np.zeros((bc, n, lda), dtype=dtype)
    for b in range(bc):
        G = g.standard_normal((n, n))
        A0[b, :, :n] = G @ G.T / n + np.eye(n)
    A0[:, :, n:] = 7
    A0[1, n // 2, n // 2] = -1  # not positive definite: info, the column below scaled by 0
    Ao = A0.copy()
    in_o = oracle.potf2(Ao, n, uplo)
    Ad = torch_gpu.from_numpy(A0).cuda()
    info = ra.potrf(handle, Ad, uplo=uplo)
    torch_gpu.cuda.synchronize()
    np.testing.assert_array_equal(info.cpu().numpy(), in_o)
    np.testing.assert_array_equal(Ad.cpu().numpy(), Ao)
