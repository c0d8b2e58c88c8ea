"""Solves of several right-hand sides round no more than solves of one: the
residuals (in extended precision) of 32 columns solved at once against those of
the same columns one by one, mean over 32 columns of 2-norms.

Bar 1.03: with sums of the same depth the two differ by chance, less than a
percent over a million components; chains twice as deep in one of the kernels
show as 4 % and more.
"""
import numpy as np
import pytest
import scipy.sparse as sps

from pastix_amd import pastix, spm
from tests.helpers import analyse

pytestmark = pytest.mark.gpu
F = pastix.factotype


def _residuals(A, x, b):
    """2-norms of b - A x, the products summed in long double."""
    xl = x.astype(np.longdouble)
    ax = np.add.reduceat(A.data.astype(np.longdouble)[:, None] * xl[A.indices, :], A.indptr[:-1], axis=0)
    return np.sqrt(((b.astype(np.longdouble) - ax) ** 2).sum(axis=0)).astype(np.float64)


@pytest.mark.parametrize("prec", [spm.SpmDouble, spm.SpmFloat])
@pytest.mark.parametrize("facto,grid", [(F.LLT, (31, 29, 34)), (F.LDLT, (31, 29, 34)), (F.LU, (24, 22, 26)),
                                        (F.LLT, (211, 197, 1)), (F.LU, (150, 140, 1))])
def test_many_as_one(facto, grid, prec):
    A = spm.convection_diffusion27(*grid, seed=1) if facto == F.LU else spm.laplacian7(*grid, diag=6.0)
    A = sps.csr_matrix(A)
    A.sort_indices()
    n = A.shape[0]
    h, S, _ = analyse(sps.csc_matrix(A), facto != F.LU, facto, grid=grid)
    pastix.set_amd_iparm(h, pastix.amd_iparm.factor_precision, prec)
    pastix.task_numfact(h, S)
    b = np.asfortranarray(np.random.default_rng(7).uniform(-1.0, 1.0, (n, 32)))
    many = b.copy(order="F")
    pastix.task_solve(h, S, many)
    one = b.copy(order="F")
    for c in range(32):
        x = np.asfortranarray(b[:, c:c + 1].copy())
        pastix.task_solve(h, S, x)
        one[:, c] = x[:, 0]
    ratio = _residuals(A, many, b).mean() / _residuals(A, one, b).mean()
    print("residuals of 32 at once / one by one:", ratio)
    assert ratio <= 1.03
    pastix.finalize(h)
