"""The staged tile products at the edges of their tiles: supernode widths
around multiples of the MFMA step (4), the staged chunk (16) and the tile
(64), odd row counts (16-byte loads that straddle the last row), against the
CPU oracle's factor.

Bar: 4500 roundings of the factor's precision, relative Frobenius (1e-12 in
FP64, the bar of the other parity tests; 2.7e-4 in FP32).
"""
import numpy as np
import pytest

from pastix_amd import pastix, spm
from tests.helpers import analyse, oracle_factor, rel_frob, lower_mask_panel

pytestmark = pytest.mark.gpu

SHAPES = [((9, 7, 5), (1, 1)), ((9, 7, 5), (3, 5)), ((31, 3, 2), (15, 17)), ((11, 11, 11), (60, 63)),
          ((13, 11, 10), (64, 65)), ((17, 16, 15), (125, 131)), ((43, 41, 1), (160, 320))]


@pytest.mark.parametrize("prec", [spm.SpmDouble, spm.SpmFloat])
@pytest.mark.parametrize("grid,bs", SHAPES)
def test_llt_tile_edges(grid, bs, prec):
    A = spm.laplacian7(*grid, coef=(1.0, 0.7, 0.4), diag=4.5)
    h, S, sym = analyse(A, True, pastix.factotype.LLT, grid=grid, min_bs=bs[0], max_bs=bs[1])
    pastix.set_amd_iparm(h, pastix.amd_iparm.factor_precision, prec)
    pastix.task_numfact(h, S)
    Lg, _ = pastix.coeftab(h, dtype=np.float64 if prec == spm.SpmDouble else np.float32)
    _, _, Lo, _ = oracle_factor(A, sym)
    err = rel_frob(lower_mask_panel(sym, Lg).astype(np.float64), lower_mask_panel(sym, Lo))
    assert err <= (1e-12 if prec == spm.SpmDouble else 2.7e-4)
    pastix.finalize(h)


@pytest.mark.parametrize("prec", [spm.SpmDouble, spm.SpmFloat])
@pytest.mark.parametrize("grid,bs", SHAPES[1:-1])
def test_lu_tile_edges(grid, bs, prec):
    A = spm.convection_diffusion27(*grid, seed=4)
    h, S, sym = analyse(A, False, pastix.factotype.LU, grid=grid, min_bs=bs[0], max_bs=bs[1])
    h.dparm[pastix.dparm.epsilon_magn_ctrl] = np.ldexp(1.0, -52)
    pastix.set_amd_iparm(h, pastix.amd_iparm.factor_precision, prec)
    pastix.task_numfact(h, S)
    Lg, Ug = pastix.coeftab(h, dtype=np.float64 if prec == spm.SpmDouble else np.float32, lu=True)
    _, _, Lo, Uo = oracle_factor(A, sym, lu=True, crit=np.ldexp(1.0, -52) * np.linalg.norm(A.data))
    bar = 1e-12 if prec == spm.SpmDouble else 2.7e-4
    assert rel_frob(Lg.astype(np.float64), Lo) <= bar and rel_frob(Ug.astype(np.float64), Uo) <= bar
    pastix.finalize(h)
