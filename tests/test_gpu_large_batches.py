"""Batches beyond one launch: HIP takes fewer than 2^32 work-items per grid
dimension, 2^23 workgroups of 512 threads, 2^25 of 128, 2^26 of 64.  Sizes are
the smallest matrices that reach the limit of each kernel; entries are small
integers and powers of two, so that the expected values are exact."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture()
def room(torch_gpu):
    torch = torch_gpu

    def need(gib):
        torch.cuda.empty_cache()
        if torch.cuda.mem_get_info()[0] < gib * 2 ** 30:
            pytest.skip(f"{gib} GiB of free device memory needed")
        return torch

    yield need
    torch.cuda.empty_cache()


def test_getrf_tall_columns(room, handle):
    """The panel's workgroup of 512 threads per matrix."""
    import rocsolver_amd as ra
    torch = room(30)
    bc, m = (1 << 23) + 5, 257
    A = torch.empty((bc, 1, m), dtype=torch.float32, device="cuda").fill_(2.0)
    row = torch.arange(bc, device="cuda") * 31 % m
    A[torch.arange(bc, device="cuda"), 0, row] = -4.0  # the pivot
    ipiv, info = ra.getrf(handle, A)
    assert int(info.abs().max()) == 0
    assert torch.equal(ipiv[:, 0].long(), row + 1)
    assert bool((A[:, 0, 0] == -4.0).all()) and bool((A[:, 0, 1:] == -0.5).all())


def test_potrf_many(room, handle):
    """64 threads per matrix."""
    import rocsolver_amd as ra
    torch = room(2)
    bc = (1 << 26) + 3
    A = torch.full((bc, 1, 1), 16.0, dtype=torch.float32, device="cuda")
    A[-1] = -1.0
    info = ra.potrf(handle, A)
    assert int(info[:-1].abs().max()) == 0 and int(info[-1]) == 1
    assert bool((A[:-1] == 4.0).all())


def test_potrs_many_systems(room, handle):
    """128 threads per system and 16 right-hand sides."""
    import rocsolver_amd as ra
    torch = room(12)
    bc, nrhs = (1 << 25) + 9, 9
    F = torch.full((bc, 1, 1), 2.0, dtype=torch.float64, device="cuda")
    B = torch.arange(bc, device="cuda").to(torch.float64)[:, None, None].repeat(1, nrhs, 1)
    ra.potrs(handle, F, B)
    assert torch.equal(B[:, 0, 0], torch.arange(bc, device="cuda").to(torch.float64) / 4)
    assert bool((B == B[:, :1]).all())


def test_potrs_many_right_hand_sides(room, handle):
    """One system, more groups of right-hand sides than a launch takes."""
    import rocsolver_amd as ra
    torch = room(6)
    nrhs = (1 << 29) - 3
    F = torch.full((1, 1, 1), 2.0, dtype=torch.float32, device="cuda")
    B = torch.full((1, nrhs, 1), 3.0, dtype=torch.float32, device="cuda")
    B[0, -1] = 5.0
    ra.potrs(handle, F, B)
    assert float(B[0, -1, 0]) == 1.25 and bool((B[0, :-1] == 0.75).all())


@pytest.mark.parametrize("trans", ["N", "T"])
def test_getrs_many_right_hand_sides(room, handle, trans):
    """The blocked solve's row interchanges: 8 right-hand sides per workgroup
    of 1024 threads."""
    import rocsolver_amd as ra
    torch = room(24)
    n, nrhs = 65, (1 << 25) + 11  # the right-hand sides exceed 2 GiB: blocked solve
    LU = (torch.eye(n, dtype=torch.float32, device="cuda") * 2).reshape(1, n, n)
    ipiv = torch.arange(n, 0, -1, dtype=torch.int32, device="cuda").clamp(min=33)[None]
    ipiv[0, 33:] = torch.arange(34, n + 1, dtype=torch.int32, device="cuda")  # rows reversed
    B = torch.empty((1, nrhs, n), dtype=torch.float32, device="cuda")
    B[:] = torch.arange(n, dtype=torch.float32, device="cuda")
    B[0, -1] += 100.0
    ra.getrs(handle, LU, ipiv, B, trans=trans)
    want = torch.arange(n - 1, -1, -1, dtype=torch.float32, device="cuda") / 2
    assert torch.equal(B[0, -1], want + 50.0)
    for c in range(0, nrhs - 1, 1 << 22):
        assert bool((B[0, c:min(nrhs - 1, c + (1 << 22))] == want).all()), c


def test_getrs_shared_factor(room, handle):
    """One factor for every system (a stride of 0): 128 threads per system."""
    import rocsolver_amd as ra
    torch = room(40)
    n, bc = 65, (1 << 25) + 5
    LU = torch.eye(n, dtype=torch.float32, device="cuda") * 2
    ipiv = torch.arange(1, n + 1, dtype=torch.int32, device="cuda")
    B = torch.full((bc, 1, n), 3.0, dtype=torch.float32, device="cuda")
    B[-1] = 5.0
    ra.check("rocsolver_sgetrs_strided_batched", handle.value, ra.OP_NONE, n, 1, LU.data_ptr(), n,
             0, ipiv.data_ptr(), 0, B.data_ptr(), n, n, bc)
    assert bool((B[-1] == 2.5).all()) and bool((B[:-1] == 1.5).all())


def test_small_systems(room, handle):
    """Four systems per wavefront: factor, solve, and factor and solve."""
    import rocsolver_amd as ra
    torch = room(16)
    bc = (1 << 28) + 5
    A = torch.full((bc, 1, 1), 4.0, dtype=torch.float32, device="cuda")
    A[-1] = 0.0
    ipiv, info = ra.getrf(handle, A)
    assert int(info[:-1].abs().max()) == 0 and int(info[-1]) == 1
    assert bool((ipiv == 1).all())
    A[-1] = 8.0
    B = torch.full((bc, 1, 1), 2.0, dtype=torch.float32, device="cuda")
    ra.getrs(handle, A, ipiv, B)
    assert bool((B[:-1] == 0.5).all()) and float(B[-1]) == 0.25
    ipiv.zero_()
    ipiv, info = ra.gesv(handle, A, B)
    assert int(info.abs().max()) == 0 and bool((ipiv == 1).all())
    assert bool((B[:-1] == 0.125).all()) and float(B[-1]) == 0.03125


def test_getri_many(room, handle):
    """A wavefront per matrix looks for zeros on the diagonal."""
    import rocsolver_amd as ra
    torch = room(4)
    bc = (1 << 26) + 3
    A = torch.full((bc, 1, 1), 4.0, dtype=torch.float32, device="cuda")
    A[-1] = 0.0
    ipiv = torch.ones((bc, 1), dtype=torch.int32, device="cuda")
    info = ra.getri(handle, A, ipiv)
    assert int(info[:-1].abs().max()) == 0 and int(info[-1]) == 1
    assert bool((A[:-1] == 0.25).all())
