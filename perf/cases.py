"""Timed cases of the solver: factorisations, solves and refinements through
the public entry points, over the sizes a program meets.

A case is a dict of plain values:
  path    "host"   pastix_task_numfact with the values of a new matrix of the
                   analysed pattern, pastix_task_solve and, when `refine` says
                   so, pastix_task_refine, all on host arrays: the calls of a
                   program written against the C API
          "device" pastix_amd_refactorize (input resident in HBM), then the
                   solve of a right-hand side block resident in HBM
          "solve"  that solve alone, on a factor made once
          "batch"  many small independent systems in one instance: numerical
                   factorisation, solve and batched refinement on host arrays
  grid    nx x ny x nz vertices (nz = 1: a 2D grid)
  stencil "lap7" (7-point Laplacian with a reaction term), "aniso7" (weights
          1, 1, 0.01), "lap5" (2D), "saddle7" (indefinite, quasi-definite
          diagonal), "cd27" (27-point convection-diffusion, nonsymmetric)
  facto   "llt", "ldlt" or "lu"
  prec    precision of the factor, "fp64" or "fp32" (of an FP64 matrix)
  refine  "" or the method that brings an FP32 factor's solution to FP64
  nrhs    right-hand sides of one call
"""
import ctypes
import functools
import math

import numpy as np
import torch

from pastix_amd import pastix, spm


def _case(name, path, grid, stencil="lap7", facto="llt", prec="fp64", refine="", nrhs=1):
    c = {"path": path, "nx": grid[0], "ny": grid[1], "nz": grid[2], "stencil": stencil, "facto": facto,
         "prec": prec, "refine": refine, "nrhs": nrhs}
    return {"name": name, **c} if name else c


def _batch_case(name, nsys, kmin, kmax):
    c = {"path": "batch", "nsys": nsys, "kmin": kmin, "kmax": kmax}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the smallest: a 20^3 grid, one numfact + solve per time step of a
        # small simulation; launches and host work count
        _case("host_llt_20x20x20", "host", (20, 20, 20)),
        # a preconditioner application: one FP32 solve of a small system
        _case("solve_fp32_24x20x18", "solve", (24, 20, 18), prec="fp32"),
        # the headline workload: 80^3 Laplacian, FP64 LL^t, refactorisation
        # from HBM and one solve
        _case("device_llt_80x80x80", "device", (80, 80, 80)),
        # the mixed-precision form of the same work on a ragged grid: FP32
        # factor, FP64 CG
        _case("device_fp32_cg_61x57x66", "device", (61, 57, 66), prec="fp32", refine="cg"),
        # nonsymmetric problems: LU of the 27-point operator
        _case("device_lu_48x48x48", "device", (48, 48, 48), stencil="cd27", facto="lu"),
        # the same through host arrays in mixed precision, GMRES
        _case("host_lu_fp32_gmres_37x41x33", "host", (37, 41, 33), stencil="cd27", facto="lu", prec="fp32",
              refine="gmres"),
        # symmetric indefinite systems, a few right-hand sides
        _case("host_ldlt_31x29x34_3rhs", "host", (31, 29, 34), stencil="saddle7", facto="ldlt", nrhs=3),
        # one solve of a kept factor: a time step with a constant operator
        _case("solve_64x64x64", "solve", (64, 64, 64)),
        # many right-hand sides of one factor: sources, load cases
        _case("solve_53x47x50_32rhs", "solve", (53, 47, 50), nrhs=32),
        # what the serving loop runs: merged requests, FP32 factor of the
        # anisotropic operator, batched CG
        _case("solve_fp32_cg_56x48x60_64rhs", "solve", (56, 48, 60), stencil="aniso7", prec="fp32", refine="cg",
              nrhs=64),
        # a large 2D problem: many narrow supernodes
        _case("device_llt_2d_701x653", "device", (701, 653, 1), stencil="lap5"),
        # small 2D systems with their own right-hand sides, in one batch
        _batch_case("batch_48_k16-128", 48, 16, 128),
    ]


def _spread(rng, lo, hi):
    """An integer in [lo, hi], its logarithm uniform."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, lo, hi):
    """A 3D grid of about lo to hi vertices, its sides within a factor of two."""
    side = _spread(rng, lo, hi) ** (1.0 / 3.0)
    return tuple(max(8, int(round(side * math.exp(rng.uniform(-0.3, 0.3))))) for _ in range(3))


def draw(rng):
    kind = rng.choice(["host", "device", "mixed", "lu", "lu_mixed", "ldlt", "solve", "solve", "serve", "grid2d",
                       "batch"])
    if kind == "host":
        return _case("", "host", _grid(rng, 4000, 60000), nrhs=_spread(rng, 1, 8))
    if kind == "device":
        return _case("", "device", _grid(rng, 8000, 250000), nrhs=_spread(rng, 1, 4))
    if kind == "mixed":
        return _case("", "device", _grid(rng, 8000, 250000), prec="fp32", refine="cg", nrhs=_spread(rng, 1, 4))
    if kind == "lu":
        return _case("", "device", _grid(rng, 4000, 100000), stencil="cd27", facto="lu", nrhs=_spread(rng, 1, 4))
    if kind == "lu_mixed":
        return _case("", "host", _grid(rng, 4000, 60000), stencil="cd27", facto="lu", prec="fp32", refine="gmres")
    if kind == "ldlt":
        return _case("", "host", _grid(rng, 4000, 50000), stencil="saddle7", facto="ldlt", nrhs=_spread(rng, 1, 8))
    if kind == "solve":
        return _case("", "solve", _grid(rng, 4000, 250000), prec=rng.choice(["fp64", "fp32"]),
                     nrhs=_spread(rng, 1, 64))
    if kind == "serve":
        return _case("", "solve", _grid(rng, 8000, 160000), stencil="aniso7", prec="fp32", refine="cg",
                     nrhs=_spread(rng, 1, 64))
    if kind == "grid2d":
        a, b = _spread(rng, 100, 700), _spread(rng, 100, 700)
        return _case("", "device", (a, b, 1), stencil="lap5", prec=rng.choice(["fp64", "fp32"]),
                     nrhs=_spread(rng, 1, 4))
    kmin = rng.randint(8, 40)
    return _batch_case("", _spread(rng, 6, 48), kmin, rng.randint(kmin + 8, 128))


# ------------------------------------------------------------------ inputs --
def _matrix(case, seed):
    """The case's matrix; the values follow the seed, the pattern does not."""
    grid = (case["nx"], case["ny"], case["nz"])
    n = grid[0] * grid[1] * grid[2]
    rng = np.random.default_rng([seed, 1])
    if case["stencil"] == "cd27":
        return spm.convection_diffusion27(*grid, seed=seed)
    q = rng.uniform(0.0, 1.0 / 16.0, n)
    if case["stencil"] == "lap7":
        A = spm.laplacian7(*grid, diag=6.0)
    elif case["stencil"] == "aniso7":
        A = spm.laplacian7(*grid, coef=(1.0, 1.0, 0.01))
    elif case["stencil"] == "lap5":
        A = spm.laplacian7(*grid, coef=(1.0, 1.0, 0.0), diag=4.0)
    else:  # saddle7: diagonally dominant, half of the diagonal negative
        A = spm.laplacian7(*grid, diag=6.5)
        sign = np.where(rng.random(n) < 0.5, -1.0, 1.0)
        A.setdiag(sign * (6.5 + q))
        return A
    A.setdiag(A.diagonal() + q)
    return A


def _solution(n, nrhs, seed, k=0):
    """The solution the right-hand sides are made from, nrhs x n."""
    return np.random.default_rng([seed, 2, k]).uniform(-1.0, 1.0, (nrhs, n))


def _systems(case, seed):
    """The batch's systems: 2D Laplacians with a shift each, 1 to 8 right-hand
    sides; sizes and counts belong to the case, values to the seed."""
    sizes = np.random.default_rng([case["nsys"], case["kmin"], case["kmax"]])
    ks = [int(k) for k in sizes.integers(case["kmin"], case["kmax"] + 1, size=case["nsys"])]
    nr = [int(r) for r in sizes.integers(1, 9, size=case["nsys"])]
    shifts = np.random.default_rng([seed, 3]).uniform(0.0, 1.0, case["nsys"])
    return ks, nr, [spm.laplacian5_2d(k, shift=float(s)) for k, s in zip(ks, shifts)]


# ------------------------------------------------------------------- state --
class _Block:
    """A torch tensor as the device buffer the entry points take."""

    def __init__(self, t):
        self.t = t
        self.ptr = ctypes.c_void_p(t.data_ptr())


class _State:
    """What a program holds: the instance, the matrix and the vectors."""

    h = None

    def __del__(self):
        if self.h is not None:
            pastix.finalize(self.h)


_FACTO = {"llt": pastix.factotype.LLT, "ldlt": pastix.factotype.LDLT, "lu": pastix.factotype.LU}


def _analysed(case, A):
    S = spm.Spm(A, symmetric=case["facto"] != "lu")
    ip, dp = pastix.initParam()
    ip[pastix.iparm.factorization] = _FACTO[case["facto"]]
    ip[pastix.iparm.ordering] = pastix.order.Personal
    ip[pastix.iparm.refinement] = pastix.refine.GMRES if case["refine"] == "gmres" else pastix.refine.CG
    dp[pastix.dparm.epsilon_refinement] = 1e-13 if case["refine"] == "cg" else 1e-12
    if case["facto"] == "lu":
        dp[pastix.dparm.epsilon_magn_ctrl] = math.ldexp(1.0, -52)
    h = pastix.init(ip, dp)
    if case["prec"] == "fp32":
        pastix.set_amd_iparm(h, pastix.amd_iparm.factor_precision, spm.SpmFloat)
    if case["path"] == "device":
        pastix.set_amd_iparm(h, pastix.amd_iparm.resident_input, 1)
    o = pastix.orderGrid(case["nx"], case["ny"], case["nz"])
    h.order = o
    pastix.subtask_order(h, S, o)
    pastix.subtask_symbfact(h)
    pastix.subtask_reordering(h)
    pastix.subtask_blend(h)
    return h, S


def _analysed_batch(mats, ks):
    S = [spm.Spm(A, symmetric=True) for A in mats]
    ip, dp = pastix.initParam()
    ip[pastix.iparm.factorization] = pastix.factotype.LLT
    ip[pastix.iparm.refinement] = pastix.refine.CG
    dp[pastix.dparm.epsilon_refinement] = 1e-13
    h = pastix.init(ip, dp)
    pastix.set_amd_iparm(h, pastix.amd_iparm.factor_precision, spm.SpmFloat)
    pastix.set_amd_iparm(h, pastix.amd_iparm.graph, 1)
    orders = [pastix.orderGrid(k, k, 1) for k in ks]
    pastix.batch_analyze(h, S, orders)
    for o in orders:
        pastix.orderExit(o)
    h.batch = None
    return h, S


def prepare(case, seed):
    st = _State()
    st.case = case
    if case["path"] == "batch":
        ks, nr, mats = _systems(case, seed)
        st.h, st.S = _analysed_batch(mats, ks)
        st.b = [np.asfortranarray(A @ _solution(A.shape[0], r, seed, i).T) for i, (A, r) in enumerate(zip(mats, nr))]
        pastix.batch_numfact(st.h, st.S)
        return st
    A = _matrix(case, seed)
    st.n = A.shape[0]
    st.h, st.S = _analysed(case, A)
    b = np.asfortranarray(A @ _solution(st.n, case["nrhs"], seed).T)
    pastix.task_numfact(st.h, st.S)
    if case["path"] == "host":
        st.b = b
        return st
    # device blocks, column-major n x nrhs: FP64 where the refinement runs,
    # the factor's precision otherwise
    dt = torch.float32 if case["prec"] == "fp32" and not case["refine"] else torch.float64
    st.b = torch.from_numpy(np.ascontiguousarray(b.T)).to("cuda", dt)
    st.x = torch.zeros_like(st.b)
    torch.cuda.synchronize()
    return st


def run(st):
    case, h = st.case, st.h
    if case["path"] == "batch":
        pastix.batch_numfact(h, st.S)
        return pastix.batch_solve_refine(h, st.b)
    if case["path"] == "host":
        pastix.task_numfact(h, st.S)
        x = st.b.copy(order="F")
        pastix.task_solve(h, st.S, x)
        if case["refine"]:
            pastix.task_refine(h, st.S, st.b, x)
        return x
    if case["path"] == "device":
        pastix.refactorize(h)
    if case["refine"]:
        pastix.solve_refine_device(h, _Block(st.b), _Block(st.x), st.n, case["nrhs"])
    else:
        # the solve works in place on its own stream: the copy comes first
        st.x.copy_(st.b)
        torch.cuda.current_stream().synchronize()
        pastix.solve_device(h, _Block(st.x), st.n, case["nrhs"])
    return st.x


def exact(case, seed):
    """The solution the right-hand sides were made from: b = A x rounds it by
    less than a condition number's worth of 2^-53."""
    if case["path"] == "batch":
        ks, nr, _ = _systems(case, seed)
        return [np.asfortranarray(_solution(k * k, r, seed, i).T) for i, (k, r) in enumerate(zip(ks, nr))]
    x = _solution(case["nx"] * case["ny"] * case["nz"], case["nrhs"], seed)
    return np.asfortranarray(x.T) if case["path"] == "host" else torch.from_numpy(x)


# -------------------------------------------------------------------- work --
# a factor larger than this leaves the chip between the forward and the
# backward sweep (256 MB of last-level cache)
_ON_CHIP = 256e6


@functools.lru_cache(maxsize=None)
def _counts(key):
    """(flops of the factorisation, entries of the factor, rows, entries of A)."""
    case = dict(key)
    if case["path"] == "batch":
        ks, _, mats = _systems(case, 0)
        h, _ = _analysed_batch(mats, ks)
        n, nnz = sum(A.shape[0] for A in mats), sum(A.nnz for A in mats)
    else:
        A = _matrix(case, 0)
        h, _ = _analysed(case, A)
        n, nnz = A.shape[0], A.nnz
    got = float(pastix.flops(h)[0]), float(h.iparm[pastix.iparm.nnzeros]), n, nnz
    pastix.finalize(h)
    return got


def work(case):
    fl, ent, n, nnz = _counts(tuple(sorted(case.items())))
    if case["path"] == "batch":
        _, nr, mats = _systems(case, 0)
        cols = sum(r * A.shape[0] for r, A in zip(nr, mats)) / n
        prec, refine, fact = "fp32", "cg", True
    else:
        cols, prec, refine, fact = case["nrhs"], case["prec"], case["refine"], case["path"] != "solve"
    size = 4 if prec == "fp32" else 8
    sweeps = 2 if ent * size > _ON_CHIP else 1
    solves = 2 if refine else 1  # the refinement applies the factor once more at least
    bytes_ = solves * sweeps * ent * size + 2 * n * cols * (8 if refine else size)
    flops = solves * 4.0 * ent * cols / (2 if case.get("facto") == "lu" else 1)
    if refine:
        bytes_ += nnz * 12
        flops += 4.0 * nnz * cols
    if fact:
        bytes_ += ent * size + nnz * 8
        flops += fl
    return {"bytes": bytes_, "flops": flops}
