"""What this framework is measured on: passes through its public entry points.

A case is a dict of plain values; `prepare` makes what a user's program holds
before the call (resident operands, plans, a kept factor), `run` is one pass
and `exact` the same result from plain torch in 64 bits.  Factorizations and
solves overwrite their operands, so a pass first restores them from device
copies (as bench.py's steps do), then calls the framework.

Kinds:
  solve    cholesky_ + ldiv_ of A = G G^T / n + I with nrhs right-hand sides
           (nrhs = 0: cholesky_ only), real or complex, 'U' or 'L'
  ldiv     ldiv_ with a factor kept on the device; nrhs = 0: a vector
  mixed    MixedCholesky (FP32 factor) + iterative refinement to 1e-13
  batched  BatchedSystems.solve over many systems of uneven size
  lu       lu_ with partial pivoting + ldiv_

PyTorch brings a HIP runtime of its own, older than the one the framework is
built with, and whichever is loaded first serves both.  In such a process
plans are issued eagerly (as the serving form and every large plan are),
never captured into a hipGraph: the older runtime does not survive the
capture of a two-stream plan.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "dagger.jl_amd"))
import dagger_mi355x as dm  # noqa: E402
from dagger_mi355x import _lib, batched, mixed  # noqa: E402

_NP = {"f64": np.float64, "f32": np.float32, "c128": np.complex128, "c64": np.complex64}
_TORCH = {"f64": torch.float64, "f32": torch.float32, "c128": torch.complex128,
          "c64": torch.complex64}
_WIDE = {"f64": torch.float64, "f32": torch.float64, "c128": torch.complex128,
         "c64": torch.complex128}
_ES = {"f64": 8, "f32": 4, "c128": 16, "c64": 8}
_REFLECTORS = 64
_PLAIN = dm.DEFAULT_OPTIONS.replace(use_graph=False)
_REFINED = _PLAIN.replace(f32_update=6, f64_diag=True)  # MixedCholesky's own, not captured


def listed():
    return [
        # the smallest request a solver service gets: one tile, pure latency
        dict(name="solve_64", kind="solve", n=64, nb=64, uplo="U", dtype="f64", nrhs=1),
        # a ragged mid-size system, cholesky!(Hermitian(A, :L)), a few right-hand sides
        dict(name="solve_1000_L", kind="solve", n=1000, nb=128, uplo="L", dtype="f64", nrhs=7),
        # the ordinary double-precision system (the configuration a CPU also runs)
        dict(name="solve_4096", kind="solve", n=4096, nb=512, uplo="U", dtype="f64", nrhs=16),
        # single precision, larger than the tuned tile grid, not a multiple of the tile
        dict(name="solve_f32_8200", kind="solve", n=8200, nb=1024, uplo="U", dtype="f32", nrhs=32),
        # complex Hermitian system (the reference's own element types)
        dict(name="solve_c128_2048", kind="solve", n=2048, nb=256, uplo="U", dtype="c128", nrhs=4),
        # the headline factorization
        dict(name="factor_32768", kind="solve", n=32768, nb=1024, uplo="U", dtype="f64", nrhs=0),
        # new right-hand sides for the headline factor kept on the device
        dict(name="ldiv_32768", kind="ldiv", n=32768, nb=1024, uplo="U", nrhs=64),
        # one new right-hand side vector for a kept factor (F \ b)
        dict(name="ldiv_vector_4096", kind="ldiv", n=4096, nb=512, uplo="U", nrhs=0),
        # low-precision factor, refined to double-precision accuracy
        dict(name="mixed_16384", kind="mixed", n=16384, nb=512, nrhs=32, kappa=1e2),
        # many small uneven systems at once, both precisions
        dict(name="batched_f64", kind="batched", count=1024, lo=32, hi=2048, mix=1, dtype="f64"),
        dict(name="batched_f32", kind="batched", count=2048, lo=32, hi=2048, mix=2, dtype="f32"),
        # a general (unsymmetric) system: LU with row pivoting
        dict(name="lu_4096", kind="lu", n=4096, nb=512, dtype="f64", nrhs=16),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _block(rng, n, smallest=64):
    fit = [b for b in (64, 128, 256, 512, 1024) if b >= smallest and b <= max(n, 64) and n <= 32 * b]
    return rng.choice(fit)


def draw(rng):
    kind = rng.choice(["solve"] * 5 + ["complex", "ldiv", "vector", "mixed", "batched", "lu"])
    if kind == "solve":
        n = _log_int(rng, 64, 12000)
        return dict(kind="solve", n=n, nb=_block(rng, n), uplo=rng.choice("UUL"),
                    dtype=rng.choice(["f64", "f64", "f32"]), nrhs=_log_int(rng, 1, 64))
    if kind == "complex":
        n = _log_int(rng, 96, 3000)
        return dict(kind="solve", n=n, nb=_block(rng, n), uplo=rng.choice("UL"),
                    dtype=rng.choice(["c128", "c64"]), nrhs=_log_int(rng, 1, 32))
    if kind == "ldiv":
        n = _log_int(rng, 512, 20000)
        return dict(kind="ldiv", n=n, nb=_block(rng, n, 128), uplo=rng.choice("UL"),
                    nrhs=_log_int(rng, 1, 64))
    if kind == "vector":
        n = _log_int(rng, 128, 8192)
        return dict(kind="ldiv", n=n, nb=_block(rng, n, 128), uplo=rng.choice("UL"), nrhs=0)
    if kind == "mixed":
        n = _log_int(rng, 1024, 16384)
        return dict(kind="mixed", n=n, nb=rng.choice([512, 1024]), nrhs=_log_int(rng, 1, 32),
                    kappa=float(10 ** rng.randint(1, 3)))
    if kind == "batched":
        return dict(kind="batched", count=rng.randint(16, 1024), lo=32,
                    hi=_log_int(rng, 128, 2048), mix=rng.randint(3, 10 ** 6),
                    dtype=rng.choice(["f64", "f32"]))
    n = _log_int(rng, 128, 5000)
    return dict(kind="lu", n=n, nb=_block(rng, n, 128), dtype=rng.choice(["f64", "f64", "f32"]),
                nrhs=_log_int(rng, 1, 32))


# ------------------------------------------------------------------ inputs
def _rng(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, cplx=False):
    if not cplx:
        return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float64)
    re = torch.randn(*shape, generator=g, device="cuda", dtype=torch.float64)
    im = torch.randn(*shape, generator=g, device="cuda", dtype=torch.float64)
    return torch.complex(re, im) * math.sqrt(0.5)


def _spd(g, n, cplx=False):
    """G G^H / n + I, exactly Hermitian."""
    G = _randn(g, n, n, cplx=cplx)
    A = G @ G.mH
    del G
    A /= n
    A.diagonal().add_(1.0)
    low = torch.tril(A, -1)
    A = torch.tril(A) + low.mH
    if cplx:
        A.imag.diagonal().zero_()
    return A


def _factor(g, n):
    """A well-conditioned upper factor with the entries a Cholesky factor of
    G G^T / n + I has: diagonal near 1.4, the rest N(0, 1/(2 n))."""
    U = torch.triu(_randn(g, n, n), 1)
    U *= math.sqrt(0.5 / n)
    U.diagonal().add_(1.2 + 0.4 * torch.rand(n, generator=g, device="cuda", dtype=torch.float64))
    return U


def _householder(g, n, kappa):
    """H diag(s) H^T with 64 reflectors and s log-spaced in [1/kappa, 1]: the
    unit vectors, s and the matrix (exactly symmetric)."""
    V = _randn(g, _REFLECTORS, n)
    V /= V.norm(dim=1, keepdim=True)
    s = kappa ** (-torch.arange(n, device="cuda", dtype=torch.float64) / max(n - 1, 1))
    A = torch.diag(s)
    for v in V.flip(0):
        A.addr_(v, v @ A, alpha=-2.0)
        A.addr_(A @ v, v, alpha=-2.0)
    low = torch.tril(A, -1)
    A = torch.tril(A) + low.T
    return V, s, A


def _operands(case, seed):
    """The dense operands of a solve/ldiv/lu case, in the case's type: A (n x n)
    and B (n x nrhs, or a vector)."""
    kind, n, nrhs = case["kind"], case["n"], case["nrhs"]
    dt = case.get("dtype", "f64")
    g = _rng(seed)
    cplx = dt in ("c64", "c128")
    if kind == "solve":
        A = _spd(g, n, cplx)
    elif kind == "ldiv":
        A = _factor(g, n)
        if case["uplo"] == "L":
            A = A.T.contiguous()
    else:
        A = _randn(g, n, n)
    B = _randn(g, n, nrhs if nrhs else 1, cplx=cplx)
    return A.to(_TORCH[dt]), B.to(_TORCH[dt])


def _mix(case):
    """Sizes (log-uniform) and right-hand-side counts of a batched case."""
    r = np.random.default_rng(case["mix"])
    n = np.exp(r.uniform(np.log(case["lo"]), np.log(case["hi"] + 1), case["count"]))
    n = np.clip(np.floor(n).astype(np.int64), case["lo"], case["hi"])
    return n, r.integers(1, 9, case["count"])


def _systems(case, seed):
    """(index, A_m, B_m) of a batched case in the case's type."""
    g = _rng(seed)
    for m, (n, r) in enumerate(zip(*_mix(case))):
        yield m, _spd(g, int(n)).to(_TORCH[case["dtype"]]), _randn(g, int(n), int(r)).to(
            _TORCH[case["dtype"]])


# ------------------------------------------------------- device arrays as torch
class _Span:
    """A device array of the framework as a torch-readable span."""

    def __init__(self, owner, ptr, count, dtype):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": np.dtype(dtype).str,
                                         "data": (ptr, False), "version": 2, "strides": None}


def _view(buffer, count, dtype):
    return torch.as_tensor(_Span(buffer, buffer.ptr, count, dtype), device="cuda")


def _flat(D):
    return _view(D.buffer, D.m * D.n, D.dtype)


def _pack(M, nb):
    """Tiles in column-major tile order, each tile column-major (the packed
    layout of a DArray)."""
    m, n = M.shape
    parts = [M[i:i + nb, j:j + nb].T.reshape(-1) for j in range(0, n, nb) for i in range(0, m, nb)]
    return torch.cat(parts)


def _upload(M, nb, vector=False):
    if vector:
        D = dm.DArray(_NP[_name(M)], (M.shape[0],), dm.Blocks(nb))
    else:
        D = dm.DArray(_NP[_name(M)], tuple(M.shape), dm.Blocks(nb, nb))
    _flat(D).copy_(_pack(M, nb))
    return D


def _name(M):
    return {v: k for k, v in _TORCH.items()}[M.dtype]


# ---------------------------------------------------------------- the passes
def prepare(case, seed):
    dm.init(torch.cuda.current_device())
    kind = case["kind"]
    st = dict(kind=kind, case=dict(case))
    if kind == "batched":
        sizes, nrhs = _mix(case)
        bs = batched.BatchedSystems(sizes, nrhs, _NP[case["dtype"]])
        _lib.call("dm_stream_sync", None)
        slab = _view(bs.A, bs.a_elems, bs.dtype)
        rhs = _view(bs.B, bs.b_elems, bs.dtype)
        for m, A, B in _systems(case, seed):
            n, ld, a0, b0 = A.shape[0], int(bs.ld[m]), int(bs.a_off[m]), int(bs.b_off[m])
            slab[a0:a0 + ld * n].view(n, ld)[:, :n].copy_(A)  # symmetric
            rhs[b0:b0 + B.numel()].copy_(B.T.reshape(-1))
        torch.cuda.synchronize()
        st.update(bs=bs, slab=slab, rhs=rhs, snap=bs.snapshot())
    elif kind == "mixed":
        g = _rng(seed)
        n, nb = case["n"], case["nb"]
        A = _householder(g, n, case["kappa"])[2]
        DA = _upload(A, nb)
        del A
        DB = _upload(_randn(g, n, case["nrhs"]), nb)
        F = dm.DArray(np.float32, (n, n), dm.Blocks(nb, nb))
        X = dm.DArray(np.float64, (n, case["nrhs"]), dm.Blocks(nb, nb))
        st.update(A=DA, B=DB, F=F, X=X)
    else:
        A, B = _operands(case, seed)
        nb = case["nb"]
        D = _upload(A, nb)
        del A
        if kind == "ldiv":
            st["F"] = dm.Cholesky(D, case["uplo"], 0)
        else:
            st["A0"], st["A"] = D, dm.DArray(D.dtype, D.shape, D.partitioning)
        if case["nrhs"] or kind == "ldiv":
            DB = _upload(B, nb, vector=not case["nrhs"])
            st["B0"], st["B"] = DB, dm.DArray(DB.dtype, DB.shape, DB.partitioning)
    torch.cuda.synchronize()
    return st


def run(st):
    kind = st["kind"]
    if kind == "batched":
        bs = st["bs"]
        bs.restore(st["snap"])
        bs.solve()
        return [st["slab"], st["rhs"], bs.infos()]
    if kind == "mixed":
        M = mixed.MixedCholesky(st["A"], options=_REFINED, F=st["F"])
        X, _ = M.solve(st["B"], tol=1e-13, max_iter=30, X=st["X"])
        return _flat(X)
    out = []
    if kind == "ldiv":
        F = st["F"]
    else:
        st["A0"].copy_into(st["A"])
        if kind == "lu":
            F = dm.lu_(st["A"], options=_PLAIN)
            out.append(F.ipiv)
        else:
            F = dm.cholesky_(st["A"], uplo=st["case"]["uplo"], options=_PLAIN)
        out.append(_flat(st["A"]))
    if "B" in st:
        st["B0"].copy_into(st["B"])
        dm.ldiv_(F, st["B"], options=_PLAIN)
        out.append(_flat(st["B"]))
    return out


# --------------------------------------------------------------- references
def work(case):
    kind = case["kind"]
    if kind == "batched":
        es = _ES[case["dtype"]]
        n, r = (v.astype(np.float64) for v in _mix(case))
        return {"bytes": float(es * (1.5 * n * n + 2 * n * r).sum()),
                "flops": float((n ** 3 / 3 + 2 * n * n * r).sum())}
    n, r = float(case["n"]), float(max(case["nrhs"], 1 if kind == "ldiv" else 0))
    es = _ES[case.get("dtype", "f64")]
    if kind == "ldiv":  # the factor's triangle, B in, X out
        return {"bytes": es * (n * n / 2 + 2 * n * r), "flops": 2 * n * n * r}
    if kind == "mixed":  # A in, X out; one factorization and one solve
        return {"bytes": 8 * (n * n + 2 * n * r), "flops": n ** 3 / 3 + 2 * n * n * r}
    if kind == "lu":
        return {"bytes": es * (2 * n * n + 2 * n * r), "flops": 2 * n ** 3 / 3 + 2 * n * n * r}
    c = 4.0 if case["dtype"] in ("c64", "c128") else 1.0
    return {"bytes": es * (1.5 * n * n + 2 * n * r), "flops": c * (n ** 3 / 3 + 2 * n * n * r)}


def _chol_solution(A, B, uplo):
    """The factor over A's triangle, as cholesky! leaves it, and the solution."""
    L = torch.linalg.cholesky(A)
    X = torch.cholesky_solve(B, L) if B.shape[1] else B
    if uplo == "U":
        return torch.triu(L.mH) + torch.tril(A, -1), X
    return torch.tril(L) + torch.triu(A, 1), X


def exact(case, seed):
    kind = case["kind"]
    if kind == "batched":
        sizes, nrhs = _mix(case)
        ld = (sizes + 1) // 2 * 2
        slab = torch.zeros(int((ld * sizes).sum()), device="cuda", dtype=torch.float64)
        rhs, a0 = [], 0
        for m, A, B in _systems(case, seed):
            n, l = A.shape[0], int(ld[m])
            F, X = _chol_solution(A.double(), B.double(), "U")
            slab[a0:a0 + l * n].view(n, l)[:, :n].copy_(F.T)
            a0 += l * n
            rhs.append(X.T.reshape(-1))
        return [slab, torch.cat(rhs), None]
    if kind == "mixed":
        g = _rng(seed)
        V, s, A = _householder(g, case["n"], case["kappa"])
        del A
        X = _randn(g, case["n"], case["nrhs"])  # B, then H diag(1/s) H^T B
        for v in V:
            X.addr_(v, v @ X, alpha=-2.0)
        X /= s[:, None]
        for v in V.flip(0):
            X.addr_(v, v @ X, alpha=-2.0)
        return _pack(X, case["nb"])
    if case["n"] > 16384 and kind != "ldiv":
        return None  # minutes in 64 bits
    A, B = _operands(case, seed)
    wide = _WIDE[case.get("dtype", "f64")]
    A, B, nb = A.to(wide), B.to(wide), case["nb"]
    if kind == "ldiv":
        U = torch.triu(A) if case["uplo"] == "U" else torch.tril(A).T
        Y = torch.linalg.solve_triangular(U.T, B, upper=False)
        X = torch.linalg.solve_triangular(U, Y, upper=True)
        return [_pack(X, nb)]
    if kind == "lu":
        LU, piv = torch.linalg.lu_factor(A.cpu())  # the host's: plain partial pivoting
        return [None, _pack(LU, nb), _pack(torch.linalg.lu_solve(LU, piv, B.cpu()), nb)]
    if not case["nrhs"]:
        return [_pack(_chol_solution(A, B[:, :0], case["uplo"])[0], nb)]
    F, X = _chol_solution(A, B, case["uplo"])
    return [_pack(F, nb), _pack(X, nb)]
