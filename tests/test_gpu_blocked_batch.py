"""A matrix's blocked LU factors do not depend on the batch it is in.

Block columns of 64 MiB or more over the batch are factored by halves, smaller
ones panel by panel; the sums are grouped by panel in both.  Tall shapes with
panels of 8 and of 16 columns, block columns in which the panels could widen,
partial last panels, columns right of the block, with and without pivoting, a
zero column in one matrix.
"""
import pytest

import rocsolver_amd as ra

pytestmark = pytest.mark.gpu

HALVES = 64 << 20  # bytes of a block column of 128 columns over the batch


@pytest.mark.parametrize("m,n", [(4096, 128), (4096, 100), (2100, 200), (1700, 130), (1600, 300), (1552, 128), (1590, 128),
                                 (2600, 100), (6000, 72), (8192, 37)])
@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("pivot", [True, False])
def test_same_bits_in_any_batch(torch_gpu, handle, m, n, dtype, pivot):
    torch = torch_gpu
    print(f"getrf {m}x{n} {dtype} pivot={pivot}", flush=True)
    dt = getattr(torch, dtype)
    few = 2
    torch.manual_seed(m + n)
    A = torch.randn(few, n, m, dtype=dt, device="cuda")
    if not pivot:
        A.diagonal(dim1=1, dim2=2).add_(3.0 * n)
    A[1, n // 2] = 0.0
    bytes_each = m * min(n, 128) * A.element_size()
    rep = -(-HALVES // (few * bytes_each)) + 1
    one, many = A.clone(), A.repeat(rep, 1, 1)
    piv1, info1 = ra.getrf(handle, one, pivot=pivot)
    piv2, info2 = ra.getrf(handle, many, pivot=pivot)
    assert torch.equal(info2.view(rep, few), info1.expand(rep, few))
    if pivot:
        assert torch.equal(piv2.view(rep, few, -1), piv1.expand(rep, few, piv1.shape[1]))
    same = (many.view(rep, few, n, m) == one) | (many.view(rep, few, n, m).isnan() & one.isnan())
    assert bool(same.all())
    # and they are factors: P A = L U within the usual bound
    if pivot:
        LU = one[0].T.double().cpu()
        L, U = torch.tril(LU, -1)[:, :min(m, n)], torch.triu(LU)[:min(m, n)]
        L += torch.eye(m, min(m, n), dtype=torch.float64)
        PA = A[0].T.double().cpu()
        for k, p in enumerate(piv1[0].tolist()):
            PA[[k, p - 1]] = PA[[p - 1, k]]
        err = (PA - L @ U).abs().max() / PA.abs().max()
        assert float(err) <= n * torch.finfo(dt).eps
