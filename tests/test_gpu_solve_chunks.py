"""Solves of more right-hand sides than one sweep takes (64), around multiples
of it and of the kernels' groups (16, 32): every column against the CPU
oracle's solve, within the engine tests' 1e-13 in FP64, and within 1e-6
normwise (17 roundings) in FP32."""
import numpy as np
import pytest

from pastix_amd import pastix, spm
from tests.helpers import analyse, oracle_factor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [spm.SpmDouble, spm.SpmFloat])
@pytest.mark.parametrize("nrhs", [48, 63, 64, 65, 80, 97, 129])
def test_chunks(nrhs, prec):
    grid = (11, 10, 9)
    A = spm.laplacian7(*grid, diag=6.0)
    h, S, sym = analyse(A, True, pastix.factotype.LLT, grid=grid, min_bs=16, max_bs=64)
    pastix.set_amd_iparm(h, pastix.amd_iparm.factor_precision, prec)
    pastix.task_numfact(h, S)
    O, _, Lo, Uo = oracle_factor(A, sym)
    p = sym["permtab"]
    _, b = spm.rhs_from_x(A, nrhs, seed=nrhs)
    x = b.copy(order="F")
    pastix.task_solve(h, S, x)
    if prec == spm.SpmDouble:
        xp = np.zeros_like(b)
        xp[p, :] = b
        xo = O.solve(Lo, Uo, xp)[p, :]
        assert (np.abs(x - xo).max(axis=0) <= 1e-13 * np.abs(xo).max(axis=0)).all()
    else:
        r = np.abs(b - A @ x).max(axis=0)
        assert (r <= 1e-6 * (abs(A).sum(axis=1).max() * np.abs(x).max(axis=0) + np.abs(b).max(axis=0))).all()
    pastix.finalize(h)
