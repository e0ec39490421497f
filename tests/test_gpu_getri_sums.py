"""The inverse without interchanges adds a block's 32 products as one sum.

One element of a triangle's inverse is 2^p (p the bits of the significand) plus
a one for each column of the blocks of 32 between: added one by one the ones are
lost (2^p + 1 rounds to 2^p), as sums of 32 they are exact.
"""
import numpy as np
import pytest

import rocsolver_amd as ra

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [65, 96, 100, 128, 129, 256, 257, 400, 512])
@pytest.mark.parametrize("upper", [False, True])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("bc", [1, 9])
def test_products_are_summed(torch_gpu, handle, n, upper, dtype, bc):
    torch = torch_gpu
    print(f"getri n={n} {dtype.__name__} upper={upper} bc={bc}", flush=True)
    big = 2.0 ** (np.finfo(dtype).nmant + 1)
    between = np.arange(32, (n - 1) // 32 * 32)
    row, col = (0, n - 1) if upper else (n - 1, 0)
    LU = np.eye(n, dtype=dtype)  # LU[column, row]
    LU[col, row] = -big
    LU[col, between] = LU[between, row] = -1
    X = np.eye(n, dtype=dtype)
    X[col, row] = big + len(between)
    X[col, between] = X[between, row] = 1
    assert X[col, row] == big + len(between)
    d = torch.from_numpy(LU).cuda().repeat(bc, 1, 1)
    ra.getri(handle, d)
    assert torch.equal(d, torch.from_numpy(X).cuda().expand_as(d))
