"""Captured device solves after the blocks that they were captured on have
moved (a later call takes more right-hand sides): the same bits as eagerly."""
import numpy as np
import pytest

from pastix_amd import pastix, spm
from tests.helpers import analyse

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [spm.SpmDouble, spm.SpmFloat])
@pytest.mark.parametrize("counts", [(1, 4, 1, 4, 9, 1), (2, 40, 2, 40, 100, 40, 2)])
def test_replays_after_more_right_hand_sides(counts, prec):
    grid = (9, 8, 7)
    A = spm.laplacian7(*grid, diag=6.0)
    n = A.shape[0]
    dt = np.float64 if prec == spm.SpmDouble else np.float32
    h, S, _ = analyse(A, True, pastix.factotype.LLT, grid=grid, min_bs=16, max_bs=40)
    pastix.set_amd_iparm(h, pastix.amd_iparm.factor_precision, prec)
    pastix.task_numfact(h, S)
    bs = {r: np.asfortranarray(spm.rhs_from_x(A, r, seed=r)[1].astype(dt)) for r in set(counts)}
    bufs = {r: pastix.DeviceArray(b) for r, b in bs.items()}

    def solve(r):
        bufs[r].upload(bs[r])
        pastix.solve_device(h, bufs[r], n, r)
        return bufs[r].download()

    # eager solves on another instance of the same factor
    g, T, _ = analyse(A, True, pastix.factotype.LLT, grid=grid, min_bs=16, max_bs=40)
    pastix.set_amd_iparm(g, pastix.amd_iparm.factor_precision, prec)
    pastix.task_numfact(g, T)
    eager = {}
    for r in bs:
        bufs[r].upload(bs[r])
        pastix.solve_device(g, bufs[r], n, r)
        eager[r] = bufs[r].download()
    pastix.set_amd_iparm(h, pastix.amd_iparm.graph, 1)
    pastix.task_numfact(h, S)
    for r in counts:
        assert np.array_equal(solve(r), eager[r]), r
    for d in bufs.values():
        d.free()
    pastix.finalize(h)
    pastix.finalize(g)
