"""Performance cases of the batched LU / Cholesky engine, through its Python entry points.

A case is a dict: ``op`` names the entry point, the rest its sizes and options.
Batches are tensors (bc, ncols, ld), each matrix column-major.  The in-place
routines overwrite their input, so a pass starts from a copy of the matrices the
program keeps, as a program that factors what it still needs does.

Distributions: float64 LU work uses N(0, 1) entries (with 0.1 n added to the
diagonal where systems are solved), float32 work the reference clients' test
matrices (integers -3..6 with about 400 on the diagonal, rows reversed, so that
every column interchanges rows), mixed-precision solves the condition numbers
1e2..1e6 of the benchmark's metric workload.
"""
import math

import numpy as np
import torch

import rocsolver_amd as ra
from rocsolver_amd import autograd as ra_autograd

_DTYPES = {"f64": torch.float64, "f32": torch.float32}
_handle = None


def _the_handle():
    """One handle for the whole program, as its users keep one."""
    global _handle
    if _handle is None:
        _handle = ra.Handle()
    return _handle


def listed():
    return [
        # a handful of tiny systems per call: launches and host work count
        dict(name="solve_small", op="gesv", dtype="f64", n=16, bc=64, nrhs=1, batched=False),
        # the many-tiny-matrices roofline (n=32 getrf of the benchmark)
        dict(name="lu_n32", op="getrf", dtype="f64", m=32, n=32, bc=131072, batched=False),
        # factor once and solve: the benchmark's n=128 configuration
        dict(name="lu_solve_n128", op="lu_solve", dtype="f64", n=128, bc=16384, nrhs=4, trans="N"),
        # single-precision solve of an odd order through the pointer-array form
        dict(name="solve_f32_n201", op="gesv", dtype="f32", n=201, bc=2500, nrhs=3, batched=True),
        # the metric workload: mixed-precision solve to float64 accuracy
        dict(name="mixed_n256", op="mixed", n=256, bc=4096, nrhs=8, factor="fp32"),
        # medium batches of large matrices, solved with the transpose
        dict(name="lu_solve_n1024", op="lu_solve", dtype="f64", n=1024, bc=64, nrhs=8, trans="T"),
        # tall panels (a block column of a larger factorisation, least squares by LU)
        dict(name="lu_tall", op="getrf", dtype="f32", m=4096, n=128, bc=64, batched=False),
        # one large system
        dict(name="solve_one_n2000", op="gesv", dtype="f64", n=2000, bc=1, nrhs=1, batched=False),
        # matrices of many orders in one call: the benchmark's variable-size batch
        dict(name="vbatch_10000", op="vbatch", dtype="f64", count=10000, lo=8, hi=512, sizes=4),
        # a differentiable solve inside a training step: forward and backward
        dict(name="grad_n96", op="grad", dtype="f64", n=96, bc=2048, nrhs=16),
        # symmetric positive definite systems (covariances)
        dict(name="posv_n300", op="posv", dtype="f64", n=300, bc=1024, nrhs=4, uplo="L"),
        # explicit inverses from the factors
        dict(name="inverse_n100", op="getri", dtype="f64", n=100, bc=2000),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _batch(rng, per, elems, hi):
    """A batch size, spread over its logarithm, of at most `elems` matrix entries."""
    return _log_int(rng, 1, max(1, min(hi, elems // per)))


def draw(rng):
    op = rng.choice(("getrf", "getrf", "gesv", "gesv", "lu_solve", "lu_solve", "mixed", "vbatch",
                     "grad", "posv", "getri"))
    dtype = rng.choice(("f64", "f64", "f32"))
    if op in ("getrf", "gesv", "lu_solve"):
        span = rng.choice(("small", "mid", "mid", "large"))
        if span == "small":
            n = _log_int(rng, 4, 64)
            bc = _batch(rng, n * n, 1 << 26, 131072)
        elif span == "mid":
            n = _log_int(rng, 65, 512)
            bc = _batch(rng, n * n, 1 << 27, 16384)
        else:
            n = _log_int(rng, 513, 1536)
            bc = _batch(rng, n * n, 1 << 25, 64)
        if op == "getrf":
            m = n
            if rng.random() < 0.4:  # rectangular, mostly tall
                m, n = _log_int(rng, 300, 4096), _log_int(rng, 16, 160)
                bc = _batch(rng, m * n, 1 << 25, 64)
                if rng.random() < 0.2:
                    m, n = n, m
            return dict(op=op, dtype=dtype, m=m, n=n, bc=bc, batched=rng.random() < 0.3)
        nrhs = rng.choice((1, 2, 3, 4, 8, 16, 25))
        if op == "gesv":
            return dict(op=op, dtype=dtype, n=n, bc=bc, nrhs=nrhs, batched=rng.random() < 0.3)
        return dict(op=op, dtype=dtype, n=n, bc=bc, nrhs=nrhs, trans=rng.choice("NT"))
    if op == "mixed":
        n = _log_int(rng, 65, 512)
        factor = rng.choice(("fp32", "fp32", "fp32", "fp16"))
        bc = _batch(rng, n * n, 1 << (27 if factor == "fp32" else 24), 8192)
        return dict(op=op, n=n, bc=bc, nrhs=rng.choice((1, 2, 5, 8)), factor=factor)
    if op == "vbatch":
        return dict(op=op, dtype=dtype, count=_log_int(rng, 100, 8000), lo=rng.randint(4, 40),
                    hi=rng.randint(64, 512), sizes=rng.randint(0, 1 << 20))
    if op == "grad":
        n = _log_int(rng, 16, 512)
        return dict(op=op, dtype=dtype, n=n, bc=_batch(rng, n * n, 1 << 24, 8192),
                    nrhs=rng.choice((1, 4, 7, 16)))
    if op == "posv":
        n = _log_int(rng, 16, 512)
        return dict(op=op, dtype=dtype, n=n, bc=_batch(rng, n * n, 3 << 24, 8192),
                    nrhs=rng.choice((1, 3, 4, 8)), uplo=rng.choice("LU"))
    n = _log_int(rng, 8, 400)
    return dict(op="getri", dtype=dtype, n=n, bc=_batch(rng, n * n, 3 << 23, 8192))


# ------------------------------------------------------------------- inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(shape, dtype, g):
    return torch.randn(shape, dtype=dtype, device="cuda", generator=g)


def _matrices(bc, m, n, dtype, g, shift):
    """(bc, n, m): n columns of m entries."""
    if dtype == torch.float32:
        A = torch.randint(-3, 7, (bc, n, m), device="cuda", generator=g).to(dtype)
        A.diagonal(dim1=1, dim2=2).add_(404.0)
        return A.flip(2).contiguous()
    A = _randn((bc, n, m), dtype, g)
    if shift:
        A.diagonal(dim1=1, dim2=2).add_(0.1 * n)
    return A


def _conditioned(bc, n, g):
    """U diag(s) V^T with s log-spaced in [1, kappa], kappa log-uniform in [1e2, 1e6]: U and V
    are one random orthogonal matrix between random signs and a reflection."""
    Q = torch.linalg.qr(torch.randn(n, n, dtype=torch.float64,
                                    generator=torch.Generator().manual_seed(n)))[0].to("cuda")
    kappa = torch.exp(torch.rand(bc, dtype=torch.float64, device="cuda", generator=g)
                      * (math.log(1e6) - math.log(1e2)) + math.log(1e2))
    t = torch.linspace(0.0, 1.0, n, dtype=torch.float64, device="cuda")
    s = torch.exp(torch.log(kappa)[:, None] * t[None, :])

    def signs():
        return torch.randint(0, 2, (bc, 1, n), device="cuda", generator=g).to(torch.float64) * 2 - 1

    M = Q[None, :, :] * s[:, None, :] * signs()  # Q D
    M = torch.matmul(M.reshape(bc * n, n), Q).reshape(bc, n, n) * signs()
    M = torch.matmul(M.reshape(bc * n, n), Q).reshape(bc, n, n)  # Q D Q D' Q
    M = M.transpose(1, 2).contiguous() * signs()
    M = torch.matmul(M.reshape(bc * n, n), Q).reshape(bc, n, n)
    u = _randn((bc, n, 1), torch.float64, g)
    u = u / u.norm(dim=1, keepdim=True)
    return (M - 2.0 * u * (u * M).sum(dim=1, keepdim=True)).contiguous()


def _sizes(case):
    r = np.random.default_rng(case["sizes"])
    n = np.rint(np.exp(r.uniform(np.log(case["lo"]), np.log(case["hi"]), size=case["count"])))
    return n.astype(np.int64), r.integers(1, 5, size=case["count"])


def _vb_fill(case, seed):
    """The flat A (U(-1, 1) + n I) and B (U(-1, 1)) of a variable-size batch, and its sizes."""
    n, nrhs = _sizes(case)
    dtype = _DTYPES[case["dtype"]]
    g = _generator(seed)
    A = torch.rand(int((n * n).sum()), dtype=dtype, device="cuda", generator=g) * 2 - 1
    B = torch.rand(int((n * nrhs).sum()), dtype=dtype, device="cuda", generator=g) * 2 - 1
    off = np.concatenate([[0], np.cumsum(n * n)[:-1]])
    first = np.concatenate([[0], np.cumsum(n)[:-1]])
    i = np.arange(int(n.sum())) - np.repeat(first, n)
    diag = torch.from_numpy(np.repeat(off, n) + i * (np.repeat(n, n) + 1)).to("cuda")
    A[diag] += torch.from_numpy(np.repeat(n, n)).to("cuda").to(dtype)
    return n, nrhs, A, B


def _inputs(case, seed):
    op = case["op"]
    g = _generator(seed)
    if op == "getrf":
        return dict(A=_matrices(case["bc"], case["m"], case["n"], _DTYPES[case["dtype"]], g, False))
    bc, n = case["bc"], case["n"]
    if op == "mixed":
        return dict(A=_conditioned(bc, n, g), B=_randn((bc, case["nrhs"], n), torch.float64, g))
    dtype = _DTYPES[case["dtype"]]
    if op == "posv":
        G = _randn((bc, n, n), dtype, g)
        A = torch.matmul(G, G.transpose(1, 2).contiguous()) / n
        A.diagonal(dim1=1, dim2=2).add_(1.0)
        return dict(A=(A + A.transpose(1, 2)) / 2, B=_randn((bc, case["nrhs"], n), dtype, g))
    got = dict(A=_matrices(bc, n, n, dtype, g, True))
    if op != "getri":
        got["B"] = _randn((bc, case["nrhs"], n), dtype, g)
    if op == "grad":
        got["dX"] = _randn((bc, case["nrhs"], n), dtype, g)
    return got


# -------------------------------------------------------------------- cases
def prepare(case, seed):
    h = _the_handle()
    if case["op"] == "vbatch":
        n, nrhs, A, B = _vb_fill(case, seed)
        vb = ra.VBatch(n, nrhs, _DTYPES[case["dtype"]])
        return dict(op="vbatch", h=h, vb=vb, A=A, B=B, case=case)
    st = dict(_inputs(case, seed), op=case["op"], h=h, case=case)
    if case["op"] == "grad":
        st["A"].requires_grad_(True)
        st["B"].requires_grad_(True)
    if case["op"] == "getri":  # the program has its factors already
        st["LU"] = st["A"].clone()
        st["ipiv"], _ = ra.getrf(h, st["LU"])
    return st


def run(st):
    op, h, case = st["op"], st["h"], st["case"]
    if op == "getrf":
        LU = st["A"].clone()
        ipiv, info = ra.getrf(h, LU, batched=case["batched"])
        return dict(LU=LU, ipiv=ipiv, info=info)
    if op == "lu_solve":
        LU, X = st["A"].clone(), st["B"].clone()
        ipiv, info = ra.getrf(h, LU)
        ra.getrs(h, LU, ipiv, X, trans=case["trans"])
        return dict(LU=LU, ipiv=ipiv, info=info, X=X)
    if op == "gesv":
        LU, X = st["A"].clone(), st["B"].clone()
        ipiv, info = ra.gesv(h, LU, X, batched=case["batched"])
        return dict(LU=LU, ipiv=ipiv, info=info, X=X)
    if op == "mixed":
        X, it, info, berr = ra.dsgesv(h, st["A"], st["B"], factor=case["factor"])
        return dict(X=X, iter=it, info=info, berr=berr)
    if op == "vbatch":
        vb = st["vb"]
        vb.A[:-1].copy_(st["A"])
        vb.B[:-1].copy_(st["B"])
        vb.gesv(h)
        return dict(LU=vb.A[:-1], X=vb.B[:-1], ipiv=vb.ipiv[:-1], info=vb.info)
    if op == "grad":
        X = ra_autograd.solve(st["A"], st["B"])
        dA, dB = torch.autograd.grad(X, (st["A"], st["B"]), st["dX"])
        return dict(X=X.detach(), dA=dA, dB=dB)
    if op == "posv":
        F, X = st["A"].clone(), st["B"].clone()
        info = ra.potrs(h, F, X, uplo=case["uplo"], posv=True)
        return dict(F=F, info=info, X=X)
    inv = st["LU"].clone()
    info = ra.getri(h, inv, st["ipiv"])
    return dict(inv=inv, info=info)


def _lu_flops(m, n):
    k = min(m, n)
    return m * n * k - (m + n) * k * k / 2.0 + k ** 3 / 3.0


def work(case):
    """Each input read once, each output written once; LAPACK operation counts times two."""
    op = case["op"]
    if op == "vbatch":
        n, nrhs = _sizes(case)
        n, nrhs = n.astype(float), nrhs.astype(float)
        es = 8 if case["dtype"] == "f64" else 4
        return {"bytes": float((2 * es * (n * n + n * nrhs) + 4 * n + 4).sum()),
                "flops": float((2 * n ** 3 / 3 + 2 * n * n * nrhs).sum())}
    es = 4 if case.get("dtype") == "f32" else 8
    bc, n = case["bc"], case["n"]
    if op == "getrf":
        m = case["m"]
        return {"bytes": bc * (2.0 * es * m * n + 4 * min(m, n) + 4), "flops": bc * 2 * _lu_flops(m, n)}
    lu = 2.0 * n ** 3 / 3
    if op == "getri":
        return {"bytes": bc * (2.0 * es * n * n + 4 * n + 4), "flops": bc * 4.0 * n ** 3 / 3}
    r = case["nrhs"]
    if op == "mixed":
        return {"bytes": bc * (8.0 * n * n + 16 * n * r + 16), "flops": bc * (lu + 2.0 * n * n * r)}
    if op == "grad":
        return {"bytes": bc * es * (2.0 * n * n + 4 * n * r), "flops": bc * (lu + 6.0 * n * n * r)}
    if op == "posv":
        return {"bytes": bc * es * (1.0 * n * n + 2 * n * r), "flops": bc * (lu / 2 + 2.0 * n * n * r)}
    return {"bytes": bc * (2.0 * es * (n * n + n * r) + 4 * n + 4), "flops": bc * (lu + 2.0 * n * n * r)}


# -------------------------------------------------------------------- exact
def _host(t):
    return t.detach().cpu().double()


def _rows(A):
    """(bc, ncols, ld) column-major -> (bc, m, n) ordinary matrices."""
    return A.transpose(1, 2).contiguous()


def _exact_lu(A):
    return torch.linalg.lu_factor(_rows(A))[0].transpose(1, 2)


def _exact_solve(A, B, transposed=False):
    M = A if transposed else _rows(A)
    return torch.linalg.solve(M, _rows(B)).transpose(1, 2).contiguous()


def exact(case, seed):
    op = case["op"]
    if op == "vbatch":
        n, nrhs, A, B = _vb_fill(case, seed)
        A, B = _host(A), _host(B)
        LU, X = torch.empty_like(A), torch.empty_like(B)
        oa = ob = 0
        for k, r in zip(n.tolist(), nrhs.tolist()):
            M = A[oa:oa + k * k].view(1, k, k)
            LU[oa:oa + k * k] = _exact_lu(M).reshape(-1)
            X[ob:ob + k * r] = _exact_solve(M, B[ob:ob + k * r].view(1, r, k)).reshape(-1)
            oa, ob = oa + k * k, ob + k * r
        return dict(LU=LU, X=X, ipiv=None, info=None)
    t = {k: _host(v) for k, v in _inputs(case, seed).items()}
    A = t["A"]
    if op == "getrf":
        return dict(LU=_exact_lu(A), ipiv=None, info=None)
    if op == "lu_solve":
        return dict(LU=_exact_lu(A), ipiv=None, info=None,
                    X=_exact_solve(A, t["B"], case["trans"] == "T"))
    if op == "gesv":
        return dict(LU=_exact_lu(A), ipiv=None, info=None, X=_exact_solve(A, t["B"]))
    if op == "mixed":
        return dict(X=_exact_solve(A, t["B"]), iter=None, info=None, berr=None)
    if op == "grad":
        X, dB = _exact_solve(A, t["B"]), _exact_solve(A, t["dX"], True)
        dA = -torch.matmul(X.transpose(1, 2).contiguous(), dB)  # dA[b, j, i] = -sum_c X[c, j] dB[c, i]
        return dict(X=X, dA=dA, dB=dB)
    if op == "posv":
        L = torch.linalg.cholesky(A)  # A = L L^T, and the buffer's rows are its columns
        F = A.triu(1) + L if case["uplo"] == "U" else A.tril(-1) + L.transpose(1, 2)
        return dict(F=F, info=None, X=_exact_solve(A, t["B"]))
    return dict(inv=torch.linalg.inv(_rows(A)).transpose(1, 2), info=None)
