"""Solves of several right-hand sides at the edges of the matrix-core kernels:
column counts around 16 and 32, node widths around 16, 32 and 64 and wider,
against the CPU oracle's solve.

Bars: FP64 within 1e-13 of the oracle's solution (the bar of the engine
tests); FP32 normwise backward error at most 1e-6 (17 roundings; FP64's bar of
1e-15 is 9).
"""
import numpy as np
import pytest

from pastix_amd import pastix, spm
from tests.helpers import analyse, oracle_factor

pytestmark = pytest.mark.gpu

SHAPES = [((9, 7, 5), (1, 1)), ((31, 3, 2), (15, 17)), ((12, 11, 10), (16, 33)), ((13, 12, 11), (60, 65)),
          ((16, 15, 14), (160, 320))]
NRHS = [2, 3, 15, 16, 17, 31, 33]


def _berr(A, x, b):
    r = b - A @ x
    return float(np.abs(r).max() / (abs(A).sum(axis=1).max() * np.abs(x).max() + np.abs(b).max()))


@pytest.mark.parametrize("facto", ["llt", "lu"])
@pytest.mark.parametrize("grid,bs", SHAPES)
def test_many_fp64(grid, bs, facto):
    lu = facto == "lu"
    A = spm.convection_diffusion27(*grid, seed=2) if lu else spm.laplacian7(*grid, diag=6.0)
    h, S, sym = analyse(A, not lu, pastix.factotype.LU if lu else pastix.factotype.LLT, grid=grid, min_bs=bs[0],
                        max_bs=bs[1])
    crit = None
    if lu:
        h.dparm[pastix.dparm.epsilon_magn_ctrl] = np.ldexp(1.0, -52)
        crit = np.ldexp(1.0, -52) * np.linalg.norm(A.data)
    pastix.task_numfact(h, S)
    O, _, Lo, Uo = oracle_factor(A, sym, lu=lu, crit=crit)
    p = sym["permtab"]
    for nrhs in NRHS:
        _, b = spm.rhs_from_x(A, nrhs, seed=nrhs)
        x = b.copy(order="F")
        pastix.task_solve(h, S, x)
        xp = np.zeros_like(b)
        xp[p, :] = b
        xo = O.solve(Lo, Uo, xp)[p, :]
        assert np.abs(x - xo).max() <= 1e-13 * np.abs(xo).max(), nrhs
    pastix.finalize(h)


@pytest.mark.parametrize("grid,bs", SHAPES)
def test_many_fp32(grid, bs):
    A = spm.laplacian7(*grid, diag=6.0)
    h, S, _ = analyse(A, True, pastix.factotype.LLT, grid=grid, min_bs=bs[0], max_bs=bs[1])
    pastix.set_amd_iparm(h, pastix.amd_iparm.factor_precision, spm.SpmFloat)
    pastix.task_numfact(h, S)
    for nrhs in NRHS:
        _, b = spm.rhs_from_x(A, nrhs, seed=nrhs)
        x = b.copy(order="F")
        pastix.task_solve(h, S, x)
        assert max(_berr(A, x[:, c], b[:, c]) for c in range(nrhs)) <= 1e-6, nrhs
    pastix.finalize(h)
