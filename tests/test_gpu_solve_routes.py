"""The row and the tile solver behind potrs and getrs agree bit for bit.

Large batches of few right-hand sides take one workgroup of rows per system,
small ones the tile solver, by tables over the order (with lines at 32-row
blocks and workgroup sizes).  A system's solution must not depend on the batch
it came in: each call on a large batch is compared with the same systems in
batches that are small enough for the tiles, and with the oracle.  Leading
dimensions exceed the order; padding rows must come back untouched.
"""
import numpy as np
import pytest

import oracle
import rocsolver_amd as ra

pytestmark = pytest.mark.gpu

FEW = 3  # distinct systems


def _factor(g, n, ld, dtype):
    F = (g.uniform(-1, 1, size=(FEW, n, ld)) / np.sqrt(n)).astype(dtype)
    F[:, np.arange(n), np.arange(n)] = g.uniform(1, 2, size=(FEW, n)).astype(dtype)
    return F


def _both(torch, call, F, B, rep):
    """The FEW systems alone and repeated `rep` times."""
    one, many = B.clone(), B.repeat(rep, 1, 1)
    call(F, one)
    call(F.repeat(rep, 1, 1), many)
    assert torch.equal(many.view(rep, *B.shape), one.expand(rep, *B.shape))
    return one.cpu().numpy()


@pytest.mark.parametrize("n", [1, 4, 5, 8, 9, 12, 20, 26, 32, 33, 44, 47, 52, 53, 64, 65, 84, 96, 97,
                               108, 127, 128, 129, 151, 224, 256, 257, 288, 384, 385, 512])
@pytest.mark.parametrize("uplo", ["L", "U"])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_potrs(torch_gpu, handle, n, uplo, dtype):
    torch = torch_gpu
    g = np.random.default_rng(n)
    F = _factor(g, n, n + 3, dtype)
    Fd = torch.from_numpy(F).cuda()
    for nrhs in (1, 3, 4, 8):
        print(f"potrs n={n} {uplo} nrhs={nrhs} {dtype.__name__}", flush=True)
        B = g.uniform(-1, 1, size=(FEW, nrhs, n + 2)).astype(dtype)
        for rep in (420, 1400) if n <= 256 else (420,):
            X = _both(torch, lambda f, b: ra.potrs(handle, f, b, uplo=uplo), Fd,
                      torch.from_numpy(B).cuda(), rep)
        Xo = B.copy()
        oracle.potrs(F, n, Xo, uplo)
        np.testing.assert_array_equal(X[:, :, n:], Xo[:, :, n:])
        err = np.abs(X - Xo).max() / np.abs(Xo).max()
        assert err <= n * np.finfo(dtype).eps


@pytest.mark.parametrize("n", [65, 76, 84, 96, 97, 104, 108, 128, 129, 136, 152, 200, 256, 257, 384, 512])
@pytest.mark.parametrize("trans", ["N", "T"])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_getrs(torch_gpu, handle, n, trans, dtype):
    torch = torch_gpu
    g = np.random.default_rng(n)
    LU = _factor(g, n, n + 3, dtype)
    ipiv = np.stack([g.integers(np.arange(1, n + 1), n + 1) for _ in range(FEW)]).astype(np.int32)
    Ld, ip = torch.from_numpy(LU).cuda(), torch.from_numpy(ipiv).cuda()

    def call(f, b):
        ra.getrs(handle, f, ip.repeat(f.shape[0] // FEW, 1), b, trans=trans)

    for nrhs in (1, 4, 8):
        print(f"getrs n={n} {trans} nrhs={nrhs} {dtype.__name__}", flush=True)
        B = g.uniform(-1, 1, size=(FEW, nrhs, n + 2)).astype(dtype)
        # beyond n = 256 in FP32 rows are taken from 513 to 768 systems and beyond 1024
        for rep in (200, 400, 800) if n > 128 else (200, 400, 1000):
            X = _both(torch, call, Ld, torch.from_numpy(B).cuda(), rep)
        Xo = B.copy()
        oracle.getrs(trans, LU, n, ipiv, Xo)
        np.testing.assert_array_equal(X[:, :, n:], Xo[:, :, n:])
        err = np.abs(X - Xo).max() / np.abs(Xo).max()
        assert err <= n * np.finfo(dtype).eps


@pytest.mark.parametrize("uplo", ["L", "U"])
def test_posv_leaves_failed_systems_alone(torch_gpu, handle, uplo):
    """B of a system whose factorisation failed is not touched by the rows."""
    torch = torch_gpu
    bc, n = 1030, 33
    A = (torch.eye(n, dtype=torch.float64, device="cuda") * 4).repeat(bc, 1, 1)
    A[500, 20, 20] = -1.0
    B = torch.ones((bc, 1, n), dtype=torch.float64, device="cuda")
    info = ra.potrs(handle, A, B, uplo=uplo, posv=True)
    assert int(info[500]) == 21 and int(info.sum()) == 21
    want = torch.full_like(B, 0.25)
    want[500] = 1.0
    assert torch.equal(B, want)
