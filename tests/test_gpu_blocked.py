"""GPU parity of the blocked LU's kernels at the edges of their dispatch, against the oracle.

The register-resident panel has one instantiation per range of row counts
(512 threads, 1 to 16 rows each, 32 to 8 columns wide), so each test runs at
the last row count of a range and the first of the next.
"""
import numpy as np
import pytest

import oracle
import rocsolver_amd as ra

pytestmark = pytest.mark.gpu
EPS = {np.float64: np.finfo(np.float64).eps, np.float32: np.finfo(np.float32).eps}
PANEL_ROWS = [65, 256, 257, 512, 513, 1024, 1025, 1536, 1537, 2048, 2049, 4096, 4097, 8192, 8193]


def rel_fro(a, b):
    return np.linalg.norm((a - b).ravel()) / max(np.linalg.norm(b.ravel()), 1e-300)


@pytest.mark.parametrize("m", PANEL_ROWS)
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_one_panel_special_values(torch_gpu, handle, m, dtype):
    """Eight columns, so one panel of any width: the same operations in the
    same order as the oracle, bit for bit, with NaN, infinities, a zero
    column, exact ties and columns that are constant."""
    print(f"panel m={m} {dtype.__name__}", flush=True)
    g = np.random.default_rng(m)
    n, bc = 8, 6
    A0 = g.uniform(-1, 1, size=(bc, n, m)).astype(dtype)
    A0[1, 3, m // 2] = np.nan
    A0[2, 0, 0] = np.nan
    A0[3, 2, m - 1] = -np.inf
    A0[4, 5, :] = 0.0
    A0[4, 1, :] = 0.5
    A0[5] = np.round(A0[5] * 4) / 4
    Ao = A0.copy()
    ip_o, in_o = oracle.getf2(Ao, m)
    Ad = torch_gpu.from_numpy(A0).cuda()
    ip, info = ra.getrf(handle, Ad, m=m)
    torch_gpu.cuda.synchronize()
    np.testing.assert_array_equal(info.cpu().numpy(), in_o)
    np.testing.assert_array_equal(ip.cpu().numpy(), ip_o)
    np.testing.assert_array_equal(Ad.cpu().numpy(), Ao)


# more columns than one outer block of 128: its last partial block, columns left and right of
# it in whole and partial chunks of 64, matrices dealt to the XCDs in groups of eight
OUTER = [(16, 700, 3), (90, 333, 9), (128, 129, 8), (513, 513, 3), (640, 640, 2), (1100, 321, 17),
         (260, 1000, 3),
         # block columns factored by halves (64 MB and more in panels of at most 16 columns)
         (4096, 128, 33), (2600, 100, 65)]


@pytest.mark.parametrize("m,n,bc", [(m, 40, 3) for m in PANEL_ROWS[1:]] + OUTER)
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_panels_and_updates(torch_gpu, handle, m, n, bc, dtype):
    """Several panels with a partial last one, lda > m: pivots equal where the
    oracle finds them unambiguous, factors within 10 min(m,n) eps there, and
    P A = L U for every matrix; the padding rows are untouched."""
    print(f"getrf m={m} n={n} bc={bc} {dtype.__name__}", flush=True)
    g = np.random.default_rng(m * 31 + n)
    lda = m + 3
    A0 = g.uniform(-1, 1, size=(bc, n, lda)).astype(dtype)
    Ao = np.ascontiguousarray(A0[:, :, :m])
    ip_o, in_o, gap = oracle.getf2(Ao, m, with_gap=True)
    Ad = torch_gpu.from_numpy(A0.copy()).cuda()
    ip, info = ra.getrf(handle, Ad, m=m, batched=True)
    torch_gpu.cuda.synchronize()
    Ag, ipg = Ad.cpu().numpy(), ip.cpu().numpy()
    np.testing.assert_array_equal(Ag[:, :, m:], A0[:, :, m:])
    Ag = np.ascontiguousarray(Ag[:, :, :m])
    np.testing.assert_array_equal(info.cpu().numpy(), in_o)
    unamb = (gap > 1e3 * max(m, n) * EPS[dtype]).all(axis=1)
    np.testing.assert_array_equal(ipg[unamb], ip_o[unamb])
    for b in np.nonzero(unamb)[0]:
        assert rel_fro(Ag[b], Ao[b]) <= 10 * min(m, n) * EPS[dtype]
    be = oracle.lu_backward_error(A0[:, :, :m].astype(np.float64), Ag.astype(np.float64), ipg, m, n,
                                  EPS[dtype])
    assert be.max() < 10.0, be


@pytest.mark.parametrize("m,n", [(300, 100), (1100, 70), (2500, 24), (530, 530)])
def test_panels_without_pivoting(torch_gpu, handle, m, n):
    g = np.random.default_rng(m)
    A0 = g.uniform(-1, 1, size=(2, n, m))
    A0[:, np.arange(n), np.arange(n)] += m
    Ao = A0.copy()
    in_o = oracle.getf2_npvt(Ao, m)
    Ad = torch_gpu.from_numpy(A0).cuda()
    _, info = ra.getrf(handle, Ad, m=m, pivot=False)
    torch_gpu.cuda.synchronize()
    np.testing.assert_array_equal(info.cpu().numpy(), in_o)
    for b in range(2):
        assert rel_fro(Ad.cpu().numpy()[b], Ao[b]) <= 10 * n * EPS[np.float64]


@pytest.mark.parametrize("n,nrhs", [(513, 1), (640, 16), (640, 17), (1000, 33), (1024, 8), (1100, 100),
                                    (2048, 3), (2049, 2), (4097, 1), (8193, 1)])
@pytest.mark.parametrize("trans", ["N", "T"])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_blocked_solve(torch_gpu, handle, n, nrhs, trans, dtype):
    """getrs beyond the fused orders on well-conditioned factors with
    arbitrary interchanges: X within n eps (relative infinity norm, the
    reference threshold) of the oracle; whole and partial tiles of 128 rows
    and of 16 / 32 right-hand sides, every range of the row permutation; the
    padding rows of B are untouched."""
    print(f"getrs n={n} nrhs={nrhs} {trans} {dtype.__name__}", flush=True)
    g = np.random.default_rng(n * 3 + nrhs)
    bc, lda, ldb = 2, n + 1, n + 5
    LU = (g.uniform(-1, 1, size=(bc, n, lda)) / n).astype(dtype)
    LU[:, np.arange(n), np.arange(n)] = g.uniform(1, 2, size=(bc, n)).astype(dtype)
    ipiv = np.stack([g.integers(np.arange(1, n + 1), n + 1) for _ in range(bc)]).astype(np.int32)
    B0 = g.uniform(-1, 1, size=(bc, nrhs, ldb)).astype(dtype)
    Xo = B0.copy()
    oracle.getrs(trans, LU, n, ipiv, Xo)
    Bd = torch_gpu.from_numpy(B0.copy()).cuda()
    ra.getrs(handle, torch_gpu.from_numpy(LU).cuda(), torch_gpu.from_numpy(ipiv).cuda(), Bd, trans=trans)
    torch_gpu.cuda.synchronize()
    Xg = Bd.cpu().numpy()
    np.testing.assert_array_equal(Xg[:, :, n:], B0[:, :, n:])
    for b in range(bc):
        err = np.abs(Xg[b, :, :n] - Xo[b, :, :n]).sum(axis=0).max()
        assert err <= n * EPS[dtype] * np.abs(Xo[b, :, :n]).sum(axis=0).max()



def test_blocked_solve_many_right_hand_sides(torch_gpu, handle):
    """More groups of right-hand sides than a grid's second dimension holds: the same 33
    columns over and over, so every copy has the solution of the first, bit for bit, and that
    one is the solution of a call with 33 columns."""
    n, copies, w = 513, 63551, 33
    print(f"getrs n={n} nrhs={copies * w}", flush=True)
    g = np.random.default_rng(7)
    LU = (g.uniform(-1, 1, size=(1, n, n)) / n).astype(np.float32)
    LU[:, np.arange(n), np.arange(n)] = g.uniform(1, 2, size=(1, n)).astype(np.float32)
    ipiv = g.integers(np.arange(1, n + 1), n + 1).astype(np.int32)[None]
    LUd, ipd = torch_gpu.from_numpy(LU).cuda(), torch_gpu.from_numpy(ipiv).cuda()
    few = torch_gpu.from_numpy(g.uniform(-1, 1, size=(1, w, n)).astype(np.float32)).cuda()
    many = few.repeat(1, copies, 1)
    ra.getrs(handle, LUd, ipd, few)
    ra.getrs(handle, LUd, ipd, many)
    torch_gpu.cuda.synchronize()
    assert torch_gpu.equal(many.view(copies, w, n), few.expand(copies, w, n))
