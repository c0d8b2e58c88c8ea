"""The level schedule on one stream and on two gives the same bits, on
problems whose levels keep all, some or none of their far updates in the main
stream (256 target tiles is the line)."""
import numpy as np
import pytest

from pastix_amd import pastix, spm
from tests.helpers import analyse

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [spm.SpmDouble, spm.SpmFloat])
@pytest.mark.parametrize("lu", [False, True])
@pytest.mark.parametrize("grid", [(6, 5, 4), (20, 19, 18), (37, 35, 33), (211, 197, 1)])
def test_one_and_two_streams(grid, lu, prec):
    A = spm.convection_diffusion27(*grid, seed=6) if lu else spm.laplacian7(*grid, diag=6.0)
    h, S, _ = analyse(A, not lu, pastix.factotype.LU if lu else pastix.factotype.LLT, grid=grid)
    pastix.set_amd_iparm(h, pastix.amd_iparm.factor_precision, prec)
    got = []
    for overlap in (0, 1):
        pastix.set_amd_iparm(h, pastix.amd_iparm.overlap, overlap)
        pastix.task_numfact(h, S)
        L, U = pastix.coeftab(h, dtype=np.float64 if prec == spm.SpmDouble else np.float32, lu=lu)
        got.append((L.copy(), U.copy() if lu else None))
    assert np.array_equal(got[0][0], got[1][0])
    assert not lu or np.array_equal(got[0][1], got[1][1])
    pastix.finalize(h)
