"""Updates from levels of narrow sources (at most 16 columns: a wave per
entry) at the edges of their pieces: source widths around the 4-column product
step, the 8-column round and the limit, 1 to over 16 rows and columns per
entry, tiles of few and of many touched columns, with and without the second
stream, against the CPU oracle's factor; and bit for bit against the product
workspace, which sums in the same order.

Bar: 4500 roundings of the factor's precision, relative Frobenius (1e-12 in
FP64, the bar of the other parity tests; 2.7e-4 in FP32).
"""
import numpy as np
import pytest

from pastix_amd import pastix, spm
from tests.helpers import analyse, oracle_factor, rel_frob, lower_mask_panel

pytestmark = pytest.mark.gpu

SHAPES = [((40, 37, 1), (1, 1)), ((61, 43, 1), (3, 5)), ((17, 14, 3), (4, 4)), ((13, 12, 11), (7, 9)),
          ((14, 13, 12), (16, 16)), ((14, 13, 12), (17, 17))]


@pytest.mark.parametrize("prec", [spm.SpmDouble, spm.SpmFloat])
@pytest.mark.parametrize("lu", [False, True])
@pytest.mark.parametrize("grid,bs", SHAPES)
def test_narrow_sources(grid, bs, lu, prec):
    A = spm.convection_diffusion27(*grid, seed=5) if lu else spm.laplacian7(*grid, coef=(1.0, 0.7, 0.4), diag=4.5)
    h, S, sym = analyse(A, not lu, pastix.factotype.LU if lu else pastix.factotype.LLT, grid=grid, min_bs=bs[0],
                        max_bs=bs[1])
    crit = None
    if lu:
        h.dparm[pastix.dparm.epsilon_magn_ctrl] = np.ldexp(1.0, -52)
        crit = np.ldexp(1.0, -52) * np.linalg.norm(A.data)
    pastix.set_amd_iparm(h, pastix.amd_iparm.factor_precision, prec)
    _, _, Lo, Uo = oracle_factor(A, sym, lu=lu, crit=crit)
    bar = 1e-12 if prec == spm.SpmDouble else 2.7e-4
    first = None
    # every level narrow: the knobs change the update's form only
    workspace = np.diff(sym["cblk_fcol"]).max() <= 16
    for overlap, ws in ((0, 0), (1, 0), (0, 1))[:3 if workspace else 2]:
        if ws:
            nl = len(pastix.level_info(h))
            pastix.set_level_knobs(h, np.zeros(nl, np.int8), np.full(nl, -1, np.int8))
        pastix.set_amd_iparm(h, pastix.amd_iparm.overlap, overlap)
        pastix.task_numfact(h, S)
        Lg, Ug = pastix.coeftab(h, dtype=np.float64 if prec == spm.SpmDouble else np.float32, lu=lu)
        if lu:
            assert rel_frob(Ug.astype(np.float64), Uo) <= bar
            assert rel_frob(Lg.astype(np.float64), Lo) <= bar
        else:
            Lg = lower_mask_panel(sym, Lg)
            assert rel_frob(Lg.astype(np.float64), lower_mask_panel(sym, Lo)) <= bar
        # the same sums in the same order in each form
        assert first is None or np.array_equal(first, Lg)
        first = Lg.copy()
    pastix.finalize(h)
