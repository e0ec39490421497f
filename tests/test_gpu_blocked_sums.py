"""Updates of the blocked LU and of the blocked solves sum at most 32 products.

A product of 2^p (p the bits of the significand) and, 32 columns on, ninety-six
ones belong to one element, from which 2^p + 96 is to be subtracted and which
holds 2^p.  A sum over all 128 columns of a block loses every one of the ones
(2^p + 1 rounds to 2^p); sums of 32 are exact, and so is what is left, -96.
"""
import numpy as np
import pytest

import rocsolver_amd as ra

pytestmark = pytest.mark.gpu

N, BLOCK = 640, 128
ONES = np.r_[32:BLOCK]


def _big(dtype):
    return 2.0 ** (np.finfo(dtype).nmant + 1)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("bc", [1, 3, 200])
@pytest.mark.parametrize("pivot", [True, False])
def test_getrf(torch_gpu, handle, dtype, bc, pivot):
    torch = torch_gpu
    print(f"getrf n={N} {dtype.__name__} bc={bc} pivot={pivot}", flush=True)
    A = np.eye(N, dtype=dtype)  # A[column, row]
    A[:BLOCK, N - 1] = 1  # L21: the row of the element
    A[N - 1, 0] = A[N - 1, N - 1] = _big(dtype)  # U12: its column
    A[N - 1, ONES] = 1
    d = torch.from_numpy(A).cuda().repeat(bc, 1, 1)
    info = ra.getrf(handle, d, pivot=pivot)[1]
    A[N - 1, N - 1] = -96
    assert not info.any()
    assert torch.equal(d, torch.from_numpy(A).cuda().expand_as(d))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nrhs,bc", [(1, 1), (20, 5), (2, 400), (64, 120), (700, 12)])
@pytest.mark.parametrize("kind", ["L", "U", "U^T", "L^T"])
def test_getrs(torch_gpu, handle, dtype, nrhs, bc, kind):
    torch = torch_gpu
    print(f"getrs n={N} {dtype.__name__} {kind} nrhs={nrhs} bc={bc}", flush=True)
    forward = kind in ("L", "U^T")
    # the block that is solved first and the element that is solved last
    cols = (0 if forward else N - BLOCK) + np.arange(BLOCK)
    i = N - 1 if forward else 0
    LU = np.eye(N, dtype=dtype)  # LU[column, row]
    LU[(i, cols) if kind.endswith("T") else (cols, i)] = 1
    B = np.zeros((nrhs, N), dtype=dtype)
    B[:, cols[0]] = B[:, i] = _big(dtype)
    B[:, cols[ONES]] = 1
    ipiv = np.arange(1, N + 1, dtype=np.int32)
    Ld, ip, d = (torch.from_numpy(x).cuda().expand(bc, *x.shape).contiguous() for x in (LU, ipiv, B))
    ra.getrs(handle, Ld, ip, d, trans="T" if kind.endswith("T") else "N")
    B[:, i] = -96
    assert torch.equal(d, torch.from_numpy(B).cuda().expand_as(d))
