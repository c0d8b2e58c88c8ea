"""A numfact's new values in every way they can come: few and many entries
(one or several host threads), one instance or a batch, FP64 and FP32, with
the analysed pattern or another one in a single system.

Bars: norms within 1e-13 of numpy's; solutions within 1e-11 of dense solves
(the bar of the batch tests).
"""
import numpy as np
import pytest
import scipy.sparse as sps

from pastix_amd import pastix, spm
from tests.helpers import analyse

F = pastix.factotype


@pytest.mark.parametrize("grid", [(3, 2, 1), (24, 23, 22), (52, 51, 50)])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_norms(grid, dtype):
    A = spm.laplacian7(*grid, diag=6.0)
    h, S, _ = analyse(A, True, F.LLT, grid=grid)
    S = spm.Spm(A, symmetric=True, dtype=dtype)
    rng = np.random.default_rng(1)
    d = sps.csc_matrix(sps.tril(A))
    cols = np.repeat(np.arange(S.n), np.diff(d.indptr))
    w = np.where(d.indices == cols, 1.0, 2.0)
    for _ in range(2):
        pastix.subtask_spm2bcsc(h, S)
        ref = np.sqrt(np.sum(w * S.values.astype(np.float64) ** 2))
        assert abs(float(h.dparm[pastix.dparm.a_norm]) - ref) <= 1e-13 * ref
        S.values[:] = (S.values * rng.uniform(0.5, 2.0, len(S.values))).astype(dtype)
    pastix.finalize(h)


def _solved(h, mats, ks):
    rng = np.random.default_rng(3)
    bs = [rng.uniform(-1.0, 1.0, (k * k, 2)) for k in ks]
    for A, b, x in zip(mats, bs, pastix.batch_solve(h, bs)):
        xd = np.linalg.solve(A.toarray(), b)
        assert np.abs(x - xd).max() <= 1e-11 * np.abs(xd).max()


@pytest.mark.gpu
@pytest.mark.parametrize("ks", [[3, 1, 7], [30, 17, 25, 40, 33] * 5 + [20] * 80])
def test_batch(ks):
    mats = [spm.laplacian5_2d(k) + (0.5 + s / len(ks)) * sps.eye(k * k) for s, k in enumerate(ks)]
    S = [spm.Spm(A, symmetric=True) for A in mats]
    ip, dp = pastix.initParam()
    ip[pastix.iparm.factorization] = F.LLT
    h = pastix.init(ip, dp)
    pastix.batch_analyze(h, S, [pastix.orderGrid(k, k, 1) for k in ks])
    pastix.batch_numfact(h, S)
    _solved(h, mats, ks)
    # new values
    mats = [A + 0.25 * sps.eye(A.shape[0]) for A in mats]
    for s, A in zip(S, mats):
        s.set_values(A)
    pastix.batch_numfact(h, S)
    _solved(h, mats, ks)
    # one system in FP32 (values exact there), one with zeros stored off the diagonal
    mats[0] = sps.csc_matrix(mats[0].astype(np.float32).astype(np.float64))
    S[0] = spm.Spm(mats[0], symmetric=True, dtype=np.float32)
    S[2].values[:] = 0.0
    S[2].values[S[2].colptr[:-1]] = 2.0
    mats[2] = sps.csc_matrix(2.0 * sps.eye(mats[2].shape[0]))
    pastix.batch_numfact(h, S)
    _solved(h, mats, ks)
    # fewer entries than analysed: refused
    S[2] = spm.Spm(mats[2], symmetric=True)
    with pytest.raises(RuntimeError):
        pastix.batch_numfact(h, S)
    pastix.finalize(h)
