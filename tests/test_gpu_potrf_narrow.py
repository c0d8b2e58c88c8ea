"""Diagonal blocks of narrow supernodes (four to a wave up to 16 columns; one to
a wave up to 32 where a level has 1024 of them) of mixed widths, with pivots
below the threshold, against the CPU oracle's factor; the count of replaced
pivots; negative pivots; and the blocks' inverses through a solve.

Bars: factor, every supernode's panel by itself, 4500 roundings of the factor's
precision (1e-12 in FP64, the bar of the other parity tests; 2.7e-4 in FP32);
solve, normwise backward error of 45 roundings (1e-14, 2.7e-6).
"""
import ctypes as ct

import numpy as np
import pytest
import scipy.sparse as sps

from pastix_amd import pastix, spm
from tests.helpers import oracle_factor

pytestmark = pytest.mark.gpu
ROOT = 20

# narrowest and widest leaf supernode, how many
SHAPES = [(1, 1, 5), (1, 16, 1), (1, 16, 38), (15, 16, 131), (16, 16, 4), (1, 32, 1030), (17, 32, 1024),
          (32, 32, 1025), (17, 32, 100)]


def _forest(lo, hi, count, scale, small, negative=False):
    """Dense leaf blocks, each coupled to three columns of a dense root; returns
    (A, block starts, columns whose pivots fall below 1e-3 scale)."""
    rng = np.random.default_rng(1000 * lo + hi + count)
    w = rng.integers(lo, hi + 1, count)
    w[0], w[-1] = lo, hi
    rang = np.concatenate([[0], np.cumsum(w)])
    n = int(rang[-1]) + ROOT
    r, c, v, tiny = [], [], [], []
    for k in range(count):
        K, f = int(w[k]), int(rang[k])
        D = np.tril(rng.uniform(-0.5, 0.5, (K + 3, K)))
        i = np.arange(K)
        D[i, i] = K + rng.uniform(1.0, 2.0, K)
        if small and k % 3 == 1:
            # every fifth column from one that moves: off its diagonal 1e-3, on
            # it 1e-4 of either sign
            t = i[i % 5 == k % 5]
            D[t, :] *= 1e-3
            D[:, t] *= 1e-3
            D[t, t] = np.where(t % 2 == 0, 1e-4, -1e-4)
            tiny += (f + t).tolist()
        if negative and k == count // 2:
            D[K - 1, K - 1] = -float(K)
        rows = np.concatenate([f + i, n - ROOT + rng.choice(ROOT, 3, replace=False)])
        R, C = np.meshgrid(rows, f + i, indexing="ij")
        keep = R >= C
        r.append(R[keep])
        c.append(C[keep])
        v.append(D[keep])
    R, C = np.tril_indices(ROOT)
    r.append(n - ROOT + R)
    c.append(n - ROOT + C)
    v.append(np.where(R == C, 4.0 * count + 10.0, 0.1))
    L = sps.coo_matrix((scale * np.concatenate(v), (np.concatenate(r), np.concatenate(c))), shape=(n, n)).tocsc()
    return sps.csc_matrix(L + sps.tril(L, -1).T), np.append(rang, n), tiny


def _analysed(A, rang, prec, thr):
    n, nb = A.shape[0], len(rang) - 1
    S = spm.Spm(A, symmetric=True)
    ip, dp = pastix.initParam()
    ip[pastix.iparm.factorization] = pastix.factotype.LLT
    ip[pastix.iparm.ordering] = pastix.order.Personal
    dp[pastix.dparm.epsilon_magn_ctrl] = -thr
    h = pastix.init(ip, dp)
    pastix.set_amd_iparm(h, pastix.amd_iparm.factor_precision, prec)
    tabs = [np.arange(n), np.arange(n), rang, np.append(np.full(nb - 1, nb - 1), -1)]
    tabs = [np.ascontiguousarray(t, dtype=np.int64) for t in tabs]
    o = pastix.pastix_order_t()
    o.vertnbr, o.cblknbr = n, nb
    o.permtab, o.peritab, o.rangtab, o.treetab = [t.ctypes.data_as(ct.POINTER(ct.c_int64)) for t in tabs]
    pastix.subtask_order(h, S, o)
    pastix.subtask_symbfact(h)
    pastix.subtask_blend(h)
    sym = pastix.symbol(h)
    assert np.array_equal(np.diff(sym["cblk_fcol"]), np.diff(rang))
    assert pastix.level_info(h)[0, 0] == nb - 1
    return h, S, sym


@pytest.mark.parametrize("prec", [spm.SpmDouble, spm.SpmFloat])
@pytest.mark.parametrize("scale", [1.0, 1e4])
@pytest.mark.parametrize("small", [False, True])
@pytest.mark.parametrize("lo,hi,count", SHAPES)
def test_factor(lo, hi, count, small, scale, prec):
    A, rang, tiny = _forest(lo, hi, count, scale, small)
    thr = 1e-3 * scale
    h, S, sym = _analysed(A, rang, prec, thr)
    pastix.task_numfact(h, S)
    assert h.iparm[pastix.iparm.static_pivoting] == len(tiny)
    Lg, _ = pastix.coeftab(h, dtype=np.float64 if prec == spm.SpmDouble else np.float32)
    _, _, Lo, _ = oracle_factor(A, sym, crit=thr)
    bar = 1e-12 if prec == spm.SpmDouble else 2.7e-4
    for c in range(sym["cblknbr"]):
        K = sym["cblk_fcol"][c + 1] - sym["cblk_fcol"][c]
        a, b = sym["cblk_coef"][c], sym["cblk_coef"][c + 1]
        P, Q = [np.tril(X[a:b].reshape((K, -1)).T.astype(np.float64)) for X in (Lg, Lo)]
        assert np.linalg.norm(P - Q) <= bar * np.linalg.norm(Q), (c, K)
    if not small:
        for nrhs in (1, 3):
            _, b = spm.rhs_from_x(A, nrhs, seed=nrhs)
            x = b.copy(order="F")
            pastix.task_solve(h, S, x)
            r = np.abs(b - A @ x).max(axis=0)
            den = abs(A).sum(axis=1).max() * np.abs(x).max(axis=0) + np.abs(b).max(axis=0)
            assert (r <= (1e-14 if prec == spm.SpmDouble else 2.7e-6) * den).all()
    pastix.finalize(h)


@pytest.mark.parametrize("prec", [spm.SpmDouble, spm.SpmFloat])
@pytest.mark.parametrize("lo,hi,count", [(1, 16, 38), (17, 32, 1024)])
def test_negative_pivot_is_reported(lo, hi, count, prec):
    A, rang, _ = _forest(lo, hi, count, 1.0, False, negative=True)
    h, S, _ = _analysed(A, rang, prec, 1e-3)
    with pytest.raises(pastix.PastixError, match="task_numfact"):
        pastix.task_numfact(h, S)
    pastix.finalize(h)
