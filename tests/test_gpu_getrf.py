"""The LU of a diagonal block at the edges of its steps (4 columns of the
elimination; 4, 8, 16, 32 columns of the joined inverses; the 64-column
block), with pivots of either sign and pivots below the threshold, against the
CPU oracle's factor and solve.

Bar: 4500 roundings of the factor's precision, relative Frobenius (1e-12 in
FP64, the bar of the other parity tests; 2.7e-4 in FP32).
"""
import numpy as np
import pytest
import scipy.sparse as sp

from pastix_amd import pastix, spm
from tests.helpers import analyse, oracle_factor, rel_frob

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [spm.SpmDouble, spm.SpmFloat])
@pytest.mark.parametrize("small", [False, True])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 8, 9, 16, 17, 31, 32, 33, 60, 63, 64, 65, 100, 131])
def test_dense_lu(n, small, prec):
    rng = np.random.default_rng(n)
    D = rng.uniform(-1.0, 1.0, (n, n))
    k = np.arange(n)
    D[k, k] = np.where(k % 3 == 0, -1.5, 1.5) * n
    if small:
        # rows and columns of size 1e-6: their pivots, 1e-12, are replaced
        s = np.where(k % 7 == 5, 1e-6, 1.0)
        D = s[:, None] * D * s[None, :]
    A = sp.csc_matrix(D)
    h, S, sym = analyse(A, False, pastix.factotype.LU, max_bs=320)
    eps = 1e-8 if small else np.ldexp(1.0, -52)
    h.dparm[pastix.dparm.epsilon_magn_ctrl] = eps
    pastix.set_amd_iparm(h, pastix.amd_iparm.factor_precision, prec)
    pastix.task_numfact(h, S)
    assert h.iparm[pastix.iparm.static_pivoting] == (np.sum(k % 7 == 5) if small else 0)
    Lg, Ug = pastix.coeftab(h, dtype=np.float64 if prec == spm.SpmDouble else np.float32, lu=True)
    O, _, Lo, Uo = oracle_factor(A, sym, lu=True, crit=eps * np.linalg.norm(A.data))
    bar = 1e-12 if prec == spm.SpmDouble else 2.7e-4
    assert rel_frob(Lg.astype(np.float64), Lo) <= bar and rel_frob(Ug.astype(np.float64), Uo) <= bar
    if not small:
        _, b = spm.rhs_from_x(A, 1, seed=n)
        x = b.copy(order="F")
        pastix.task_solve(h, S, x)
        p = sym["permtab"]
        xp = np.zeros_like(b)
        xp[p, :] = b
        assert rel_frob(x, O.solve(Lo, Uo, xp)[p, :]) <= bar
    pastix.finalize(h)
