"""Blocked solves with many right-hand sides in large batches.

They take updates in launches of their own and up to 128 right-hand sides per
workgroup; few right-hand sides or systems take update and solve in one launch
per 128 rows.  The same sums in both: a right-hand side's solution must not
depend on its company, bit for bit, and must agree with the oracle.
"""
import numpy as np
import pytest

import oracle
import rocsolver_amd as ra

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [513, 640, 700, 1025])
@pytest.mark.parametrize("trans", ["N", "T"])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nrhs,bc", [(16, 300), (17, 300), (64, 120), (65, 100), (129, 64), (1500, 6),
                                     (200, 120)])
def test_same_bits(torch_gpu, handle, n, trans, dtype, nrhs, bc):
    torch = torch_gpu
    print(f"getrs n={n} {trans} {dtype.__name__} nrhs={nrhs} bc={bc}", flush=True)
    g = np.random.default_rng(n + nrhs)
    few, lda, ldb = 2, n + 3, n + 1
    LU = (g.uniform(-1, 1, size=(few, n, lda)) / np.sqrt(n)).astype(dtype)
    LU[:, np.arange(n), np.arange(n)] += np.asarray(2, dtype)
    ipiv = np.stack([g.integers(np.arange(1, n + 1), n + 1) for _ in range(few)]).astype(np.int32)
    B = g.uniform(-1, 1, size=(few, nrhs, ldb)).astype(dtype)
    Ld, ip, Bd = (torch.from_numpy(x).cuda() for x in (LU, ipiv, B))
    many = Bd.repeat(bc // few, 1, 1)
    ra.getrs(handle, Ld.repeat(bc // few, 1, 1), ip.repeat(bc // few, 1), many, trans=trans)
    many = many.view(bc // few, few, nrhs, ldb)
    assert torch.equal(many, many[:1].expand_as(many))
    cols = sorted({0, 1, nrhs // 2, nrhs - 1})
    alone = Bd[:, cols].contiguous()
    ra.getrs(handle, Ld, ip, alone, trans=trans)
    assert torch.equal(many[0][:, cols], alone)  # padding rows included
    Xo = B[:, cols].copy()
    oracle.getrs(trans, LU, n, ipiv, Xo)
    err = np.abs(alone.cpu().numpy() - Xo).max() / np.abs(Xo).max()
    assert err <= n * np.finfo(dtype).eps


def test_singular_systems_keep_their_right_hand_sides(torch_gpu, handle):
    """gesv leaves B of a singular system alone in the separate updates too."""
    torch = torch_gpu
    n, nrhs, bc = 520, 100, 64
    A = (torch.eye(n, dtype=torch.float64, device="cuda") * 2).repeat(bc, 1, 1)
    A[7, 100] = 0.0
    B = torch.ones((bc, nrhs, n), dtype=torch.float64, device="cuda")
    _, info = ra.gesv(handle, A, B)
    assert int(info[7]) == 101 and int(info.sum()) == 101
    want = torch.full_like(B, 0.5)
    want[7] = 1.0
    assert torch.equal(B, want)
