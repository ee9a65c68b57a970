"""Performance cases of the framework: the work its users have it do, through
its public entry points (starpu_amd.runtime, starpu_amd.batched and
starpu_amd.kernels), on one MI355X.

  tile     the four tile operations a StarPU codelet calls on its stream:
           POTRF of a diagonal tile (with the inverses the panel and the
           solves multiply by), TRSM, SYRK and GEMM of its neighbours
  dag      FP64 factor and solve of one system as a tile task graph
  solve    new right-hand sides on a resident FP64 factor
  mixed    low-precision factor with FP64 iterative refinement
  batch    many small systems of uneven sizes, FP64, in one launch
  batch_ir the same with an FP32 factor and FP64 refinement
  serve    the solve server on a queue of requests, a part of them re-solves

Matrices are A = G G^T / n + shift I with G i.i.d. N(0, 1), symmetric, made by
torch on the GPU from the seed; a row-major torch matrix is its own
column-major transpose, so a factor comes back in the upper triangle of the
torch view, and right-hand sides are the rows of an (nrhs, n) tensor.
"""
from __future__ import annotations

import math
import os
import tempfile

import numpy as np
import torch

from starpu_amd import batched
from starpu_amd import kernels as K
from starpu_amd import runtime as R

FP64 = torch.float64
_rt = None


# ------------------------------------------------------------------ cases

def listed():
    return [
        # a small tile: every launch counts (tile 256 is the CPU configuration's)
        {"name": "tile 256", "kind": "tile", "nb": 256},
        # the tile of the reference's own performance models
        {"name": "tile 960", "kind": "tile", "nb": 960},
        # one small system: 8 x 8 tiles of 256, one right-hand side
        {"name": "dag 2048", "kind": "dag", "n": 2048, "nb": 256, "nrhs": 1},
        # an ordinary system whose size is no multiple of anything
        {"name": "dag 6001", "kind": "dag", "n": 6001, "nb": 512, "nrhs": 5},
        # the headline system: 32 x 32 tiles of 1024, 16 right-hand sides
        {"name": "dag 32768", "kind": "dag", "n": 32768, "nb": 1024, "nrhs": 16},
        # a resident factor with new right-hand sides
        {"name": "solve 16384", "kind": "solve", "n": 16384, "nb": 1024, "nrhs": 16},
        # the two update precisions on the ill-conditioned matrix (cond ~4e3)
        {"name": "mixed bf16x3 32768", "kind": "mixed", "n": 32768, "nb": 1024, "nrhs": 16, "prec": "bf16x3"},
        {"name": "mixed fp32 6144", "kind": "mixed", "n": 6144, "nb": 512, "nrhs": 5, "prec": "fp32"},
        # a handful of small systems of odd sizes
        {"name": "batch 24 odd", "kind": "batch", "nsys": 24, "nmin": 5, "nmax": 333, "nrhs": 3},
        # the large batch: 2048 systems of 32, 64, ..., 1024
        {"name": "batch 2048", "kind": "batch", "nsys": 2048, "nmin": 32, "nmax": 1024, "nrhs": 1},
        {"name": "batch_ir 2048", "kind": "batch_ir", "nsys": 2048, "nmin": 32, "nmax": 1024, "nrhs": 1},
        # requests of mixed sizes, all waiting, 4 served at once
        {"name": "serve 32", "kind": "serve", "nreq": 32, "nmin": 256, "nmax": 8192, "nb": 512, "prec": "fp32"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tile", "dag", "solve", "mixed", "batch", "batch_ir", "serve"])
    if kind == "tile":
        return {"kind": kind, "nb": _log(rng, 64, 2048)}
    if kind in ("dag", "solve", "mixed"):
        n = _log(rng, 768, 24576)
        if rng.random() < 0.5:
            n = max(512, 128 * round(n / 128))
        nb = rng.choice([256, 512] if n < 4096 else [512, 1024])
        case = {"kind": kind, "n": n, "nb": nb, "nrhs": _log(rng, 1, 32)}
        if kind == "mixed":
            case["n"] = min(n, 16384)
            case["prec"] = rng.choice(["bf16x3", "fp32"])
        return case
    if kind in ("batch", "batch_ir"):
        nmin = rng.randrange(1, 65)
        return {"kind": kind, "nsys": _log(rng, 8, 1024), "nmin": nmin, "nmax": nmin + _log(rng, 16, 960),
                "nrhs": rng.choice([1, 1, 2, 3, 5])}
    return {"kind": kind, "nreq": rng.randrange(8, 33), "nmin": 256, "nmax": _log(rng, 1024, 6144),
            "nb": rng.choice([256, 512]), "prec": rng.choice(["fp32", "bf16x3"])}


# ----------------------------------------------------------------- inputs

def _gen(seed, part=0):
    return torch.Generator(device="cuda").manual_seed(1000003 * int(seed) + part)


def _randn(gen, *shape):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=FP64)


def _spd(gen, n, shift, count=None):
    """A (or `count` of them): G G^T / n + shift I, the two triangles equal."""
    G = _randn(gen, n, n) if count is None else _randn(gen, count, n, n)
    A = torch.matmul(G, G.mT.contiguous())
    del G
    A.mul_(1.0 / n)
    for i in range(0, n, 4096):                   # by blocks of rows: no second matrix
        j = min(n, i + 4096)
        blk = A[..., i:j, i:j]
        blk.copy_(blk.triu() + blk.triu(1).mT)
        A[..., j:, i:j] = A[..., i:j, j:].mT
    A.diagonal(dim1=-2, dim2=-1).add_(shift)
    return A


_SHIFT = {"tile": 1.0, "dag": 1.0, "solve": 1.0, "mixed": 1e-3, "batch": 0.1, "batch_ir": 0.1, "serve": 0.01}


def _system(case, seed):
    """(A, B): the matrix and its right-hand sides, one a row."""
    gen = _gen(seed)
    n = case["n"]
    return _spd(gen, n, _SHIFT[case["kind"]]), _randn(gen, case["nrhs"], n)


def _tile_inputs(case, seed):
    gen = _gen(seed)
    nb = case["nb"]
    D = _spd(gen, nb, _SHIFT["tile"])
    return D, _randn(gen, nb, nb), _randn(gen, nb, nb), _randn(gen, nb, nb)


def _batch_sizes(case):
    """At most 32 different sizes, evenly spread over the range, in a mixed
    order that the case fixes."""
    lo, hi = case["nmin"], case["nmax"]
    m = min(32, hi - lo + 1)
    levels = np.round(np.linspace(lo, hi, m)).astype(int) if m > 1 else np.array([lo])
    pick = np.random.default_rng(case["nsys"]).integers(0, m, case["nsys"])
    pick[: min(m, 2)] = [m - 1, 0][: min(m, 2)]   # the largest and the smallest are always there
    return [int(levels[p]) for p in pick]


def _batch_inputs(case, seed):
    """(sizes, {size: (systems of that size, their matrices, their right-hand sides)})."""
    sizes = _batch_sizes(case)
    groups = {}
    for v in sorted(set(sizes)):
        gen = _gen(seed, v)
        idx = [i for i, s in enumerate(sizes) if s == v]
        groups[v] = (idx, _spd(gen, v, _SHIFT[case["kind"]], len(idx)), _randn(gen, len(idx), case["nrhs"], v))
    return sizes, groups


def _offsets(sizes, per):
    off, at = [], 0
    for v in sizes:
        off.append(at)
        at += per(v)
    return off, at


def _trace(case):
    """[(n, nrhs, matrix)] of the requests: N log-uniform, a multiple of 256;
    3 in 10 requests take an earlier request's matrix."""
    rng = np.random.default_rng(case["nreq"])
    got, matrices = [], []
    for _ in range(case["nreq"]):
        if matrices and rng.random() < 0.3:
            m = int(rng.integers(0, len(matrices)))
        else:
            v = math.exp(rng.uniform(math.log(case["nmin"]), math.log(case["nmax"])))
            matrices.append(int(min(case["nmax"], max(case["nmin"], 256 * round(v / 256)))))
            m = len(matrices) - 1
        got.append((matrices[m], int(rng.integers(1, 33)), m))
    return got, matrices


# ------------------------------------------------------------------- runs

def _runtime():
    """The runtime as a program starts it once: one GPU, 12 streams, dmda, its
    calibration files in a directory of their own."""
    global _rt
    if _rt is None:
        _rt = tempfile.TemporaryDirectory(prefix="starpu_perfmodels_")
        for name in ("STARPU_HIP_RESERVE_CUS", "STARPU_CALIBRATE", "STARPU_LIMIT_HIP_MEM"):
            os.environ.pop(name, None)
        R.init(STARPU_NHIP=1, STARPU_NCPU=0, STARPU_SCHED="dmda", STARPU_NWORKER_PER_HIP=12,
               STARPU_PERF_MODEL_DIR=_rt.name)
    return R.hip_node(0)


class _Device:
    """A framework array as torch sees one."""

    def __init__(self, d, count, typestr):
        self.owner = d
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": typestr, "data": (d.ptr, False),
                                         "strides": None, "version": 2}


def _view(d, count, typestr="<f8"):
    return torch.as_tensor(_Device(d, count, typestr), device="cuda")


def prepare(case, seed):
    kind = case["kind"]
    if kind == "tile":
        D, P, Q, C = _tile_inputs(case, seed)
        e = torch.empty_like
        st = {"D0": D, "P0": P, "Q": Q, "C0": C, "L": e(D), "P": e(P), "S": e(D), "C": e(C), "W": e(D), "Linv": e(D),
              "info": torch.zeros(1, dtype=torch.int32, device="cuda")}
    elif kind in ("dag", "solve", "mixed"):
        A, B = _system(case, seed)
        st = {"A": A, "B": B, "X": torch.empty_like(B), "node": _runtime(),
              "nblocks": max(1, round(case["n"] / case["nb"]))}
        if kind == "solve":
            st["L"] = torch.linalg.cholesky(A).mT.contiguous()
            del st["A"]
        elif kind == "dag":
            st["L"] = torch.empty_like(A)
    elif kind in ("batch", "batch_ir"):
        sizes, groups = _batch_inputs(case, seed)
        b = batched.Batch(sizes, nrhs=case["nrhs"], shift=1.0, seed=1, ir=(kind == "batch_ir"))
        A0, B0 = _view(b.A0, b.totA), _view(b.B0, b.totB)
        for v, (idx, A, B) in groups.items():
            for q, i in enumerate(idx):
                A0[b.offA[i]: b.offA[i] + v * v] = A[q].reshape(-1)
                B0[b.offB[i]: b.offB[i] + v * case["nrhs"]] = B[q].reshape(-1)
        torch.cuda.synchronize()
        b.restore()
        K.sync()
        st = {"batch": b, "info": _view(b.info, b.nsys, "<i4")}
        if kind == "batch":
            st.update(A=_view(b.A, b.totA), B=_view(b.B, b.totB))
        else:
            st["X"] = _view(b.X, b.totB)
    else:
        trace, matrices = _trace(case)
        mats = [_spd(_gen(seed, m), n, _SHIFT["serve"]) for m, n in enumerate(matrices)]
        gen = _gen(seed, 10 ** 6)
        off, tot = _offsets([n * r for n, r, _ in trace], lambda v: v)
        B = _randn(gen, tot)
        X = torch.empty_like(B)
        reqs = (R.ServeRequest * len(trace))()
        for q, (n, r, m), o in zip(reqs, trace, off):
            q.n, q.nrhs, q.matrix, q.arrival_us = n, r, m, 0.0
            q.A, q.lda = mats[m].data_ptr(), n
            q.B, q.ldb, q.X, q.ldx = B.data_ptr() + 8 * o, n, X.data_ptr() + 8 * o, n
        cfg = R.ServeConfig()
        cfg.budget_bytes, cfg.slots, cfg.nb, cfg.prec = 60e9, 4, case["nb"], R.PREC[case["prec"]]
        cfg.maxiter, cfg.prio, cfg.tol = 40, 1, 1e-14
        st = {"mats": mats, "B": B, "X": X, "reqs": reqs, "cfg": cfg, "node": _runtime()}
    st["case"] = case
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "tile":
        nb = case["nb"]
        p = {k: v.data_ptr() for k, v in st.items() if isinstance(v, torch.Tensor)}
        # a codelet works in place on its tiles: they start from the inputs
        for name, src in (("L", "D0"), ("P", "P0"), ("S", "D0"), ("C", "C0")):
            st[name].copy_(st[src])
        K.dpotrf_tile(nb, p["L"], nb, p["Linv"], nb, p["W"], nb, p["info"])
        K.dtrsm_rltn(nb, nb, 1.0, p["L"], nb, p["P"], nb)
        K.dsyrk_ln(nb, nb, -1.0, p["P"], nb, 1.0, p["S"], nb)
        K.dgemm_nt(nb, nb, nb, -1.0, p["Q"], nb, p["P"], nb, 1.0, p["C"], nb)
        return {k: st[k] for k in ("L", "W", "Linv", "P", "S", "C", "info")}
    if kind == "dag":
        n = case["n"]
        st["L"].copy_(st["A"])
        st["X"].copy_(st["B"])
        K.sync()                                  # the runtime's streams start from finished inputs
        s = R.factor_solve(st["L"].data_ptr(), n, n, st["nblocks"], st["X"].data_ptr(), n, case["nrhs"],
                           home_node=st["node"])
        return {"L": st["L"], "X": st["X"], "info": s.info}
    if kind == "solve":
        n = case["n"]
        st["X"].copy_(st["B"])
        K.sync()
        R.solve(st["L"].data_ptr(), n, n, st["nblocks"], st["X"].data_ptr(), n, case["nrhs"], home_node=st["node"])
        return {"X": st["X"]}
    if kind == "mixed":
        n = case["n"]
        s = R.mixed_solve(st["A"].data_ptr(), n, n, st["nblocks"], st["B"].data_ptr(), n, case["nrhs"],
                          st["X"].data_ptr(), n, prec=case["prec"], hip_node=st["node"], prio="parsec")
        return {"X": st["X"], "info": s.info, "converged": s.converged}
    if kind == "batch":
        st["batch"].restore()                     # factored in place: the systems come in anew
        st["batch"].launch(512)
        return {"A": st["A"], "X": st["B"], "info": st["info"]}
    if kind == "batch_ir":
        st["batch"].launch_ir(512)
        return {"X": st["X"], "info": st["info"]}
    R.serve(st["cfg"], st["reqs"], hip_node=st["node"])
    return {"X": st["X"], "status": [q.status for q in st["reqs"]]}


# ------------------------------------------------------------------- work

def work(case):
    """The least a pass can do: a matrix counts once in and once out where it
    is overwritten (its lower triangle), flops as LAPACK counts them; the
    refinement's own steps are the method's, not the result's, and are left
    out but for one residual and one solve."""
    kind = case["kind"]
    if kind == "tile":
        v = float(case["nb"])
        # potrf + inverse, trsm, syrk, gemm; D, P, Q, C in, L, W, Linv, P, S, C out
        return {"flops": 2 * v ** 3 / 3 + v ** 3 + v ** 3 + 2 * v ** 3, "bytes": 8 * v * v * (0.5 + 1 + 0.5 + 2 + 5)}
    if kind in ("dag", "solve", "mixed"):
        v, r = float(case["n"]), case["nrhs"]
        fact = 0.0 if kind == "solve" else v ** 3 / 3
        tri = 4 * v * v
        return {"flops": fact + 2 * v * v * r * (2 if kind == "mixed" else 1),
                "bytes": tri * (2 if kind == "dag" else 1) + 16 * v * r}
    if kind in ("batch", "batch_ir"):
        s = np.array(_batch_sizes(case), dtype=np.float64)
        return {"flops": float(np.sum(s ** 3 / 3 + 2 * s * s * case["nrhs"])),
                "bytes": float(np.sum((8 if kind == "batch" else 4) * s * s + 16 * s * case["nrhs"]))}
    trace, matrices = _trace(case)
    return {"flops": sum(float(n) ** 3 / 3 for n in matrices) + sum(4.0 * n * n * r for n, r, _ in trace),
            "bytes": sum(4.0 * n * n for n in matrices) + sum(16.0 * n * r for n, r, _ in trace)}


# -------------------------------------------------------------- tolerance

def tolerance(case):
    kind = case["kind"]
    if kind in ("tile", "dag", "solve", "batch"):
        # FP64 throughout: 2e-16 to 1.3e-15 from the 64-bit reference at
        # condition numbers of about 5, a few times that at the batch's 40
        return {"rel": 5e-14, "max": 5e-12} if kind == "batch" else {"rel": 1e-14, "max": 1e-12}
    # refined until ||r|| <= 1e-14 (||A||_F ||x|| + ||b||), so the solution is
    # off by up to 1e-14 cond(A) ||A||_F / ||A||_2 (cond(A) about 40 for
    # batch_ir, 400 for serve, 4000 for mixed, the ratio sqrt(n) / 3): which
    # step is the last, and how far below the bound it ends, turns on the
    # factor's rounding (1e-11 and 1e-13 seen for mixed)
    return {"batch_ir": {"rel": 1e-11, "max": 1e-9}, "serve": {"rel": 1e-10, "max": 1e-8},
            "mixed": {"rel": 1e-9, "max": 1e-7}}[kind]


# ------------------------------------------------------------------ exact

def _chol_solve(A, B):
    """(L, X) of A X = B with one right-hand side a row of B."""
    L = torch.linalg.cholesky(A)
    return L, torch.cholesky_solve(B.mT, L).mT


def exact(case, seed):
    kind = case["kind"]
    if kind == "tile":
        D, P, Q, C = _tile_inputs(case, seed)
        L = torch.linalg.cholesky(D)
        inv = torch.linalg.solve_triangular(L, torch.eye(case["nb"], dtype=FP64, device="cuda"), upper=False)
        # P holds the column-major panel's transpose: (P^T L^-T)^T = L^-1 P
        Pn = torch.linalg.solve_triangular(L, P, upper=False)
        S = torch.triu(D - Pn.mT @ Pn) + torch.tril(D, -1)
        return {"L": torch.triu(L.mT) + torch.tril(D, -1), "W": inv, "Linv": inv.mT.contiguous(), "P": Pn, "S": S,
                "C": C - Pn.mT @ Q, "info": None}
    if kind in ("dag", "solve", "mixed"):
        A, B = _system(case, seed)
        L, X = _chol_solve(A, B)
        if kind == "dag":
            n = case["n"]
            L = L.mT.contiguous()
            for i in range(0, n, 4096):
                j = min(n, i + 4096)
                L[i:j, i:j] = torch.triu(L[i:j, i:j]) + torch.tril(A[i:j, i:j], -1)
                L[j:, i:j] = A[j:, i:j]
            return {"L": L, "X": X, "info": None}
        return {"X": X} if kind == "solve" else {"X": X, "info": None, "converged": None}
    if kind in ("batch", "batch_ir"):
        sizes, groups = _batch_inputs(case, seed)
        r = case["nrhs"]
        offA, totA = _offsets(sizes, lambda v: v * v)
        offB, totB = _offsets(sizes, lambda v: v * r)
        # on the CPU: torch's batched factorisation of large batches fails on the GPU
        Aout = torch.empty(totA if kind == "batch" else 1, dtype=FP64)
        Xout = torch.empty(totB, dtype=FP64)
        for v, (idx, A, B) in groups.items():
            A = A.cpu()
            L, X = _chol_solve(A, B.cpu())
            for q, i in enumerate(idx):
                if kind == "batch":
                    F = Aout[offA[i]: offA[i] + v * v].view(v, v)
                    torch.triu(L[q].mT, out=F)
                    F += torch.tril(A[q], -1)
                Xout[offB[i]: offB[i] + v * r] = X[q].reshape(-1)
        return {"A": Aout, "X": Xout, "info": None} if kind == "batch" else {"X": Xout, "info": None}
    trace, matrices = _trace(case)
    factors = [torch.linalg.cholesky(_spd(_gen(seed, m), n, _SHIFT["serve"])) for m, n in enumerate(matrices)]
    off, tot = _offsets([n * r for n, r, _ in trace], lambda v: v)
    B = _randn(_gen(seed, 10 ** 6), tot)
    X = torch.empty_like(B)
    for (n, r, m), o in zip(trace, off):
        X[o: o + n * r] = torch.cholesky_solve(B[o: o + n * r].view(r, n).mT, factors[m]).mT.reshape(-1)
    return {"X": X, "status": None}
