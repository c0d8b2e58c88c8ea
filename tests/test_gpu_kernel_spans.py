"""Timed spans of the single-pass multi-source updates: one per kernel launch
(LL^t: the tiles of few columns and the others, those of the next level and the
later ones, each in a launch of its own; LU: either side)."""
import ctypes as ct

import numpy as np
import pytest
import scipy.sparse as sps

from pastix_amd import pastix, spm

pytestmark = pytest.mark.gpu
F = pastix.factotype


def _arrow(root, rows):
    """One-column supernodes with entries in the given rows of a dense block of
    `root` columns (filled by its first one, which couples to all)."""
    k = len(rows)
    r = [np.arange(k + root)] + [k + np.asarray(x) for x in rows] + [k + np.arange(1, root)]
    c = [np.arange(k + root)] + [np.full(len(x), j) for j, x in enumerate(rows)] + [np.full(root - 1, k)]
    r, c = np.concatenate(r), np.concatenate(c)
    L = sps.coo_matrix((np.where(r == c, 1e4, 1.0), (r, c)), shape=(k + root, k + root))
    return sps.csc_matrix(L + sps.tril(L, -1).T)


WIDE, FEW = list(range(1, 41)), [130, 131, 132]


@pytest.mark.parametrize("facto", [F.LLT, F.LU])
@pytest.mark.parametrize("rows,launches", [([FEW] * 5, 1), ([WIDE] * 5, 1), ([WIDE] * 5 + [FEW] * 5, 2),
                                           ([FEW], 0)])
def test_spans_of_a_narrow_level(rows, launches, facto):
    root = 300
    A = _arrow(root, rows)
    n, k = A.shape[0], len(rows)
    S = spm.Spm(A, symmetric=facto == F.LLT)
    ip, dp = pastix.initParam()
    ip[pastix.iparm.factorization] = facto
    ip[pastix.iparm.ordering] = pastix.order.Personal
    ip[pastix.iparm.min_blocksize] = 16
    ip[pastix.iparm.max_blocksize] = 400
    h = pastix.init(ip, dp)
    tabs = [np.arange(n), np.arange(n), np.append(np.arange(k + 1), n), np.append(np.full(k, k), -1)]
    tabs = [np.ascontiguousarray(t, dtype=np.int64) for t in tabs]
    o = pastix.pastix_order_t()
    o.vertnbr, o.cblknbr = n, k + 1
    o.permtab, o.peritab, o.rangtab, o.treetab = [t.ctypes.data_as(ct.POINTER(ct.c_int64)) for t in tabs]
    pastix.subtask_order(h, S, o)
    pastix.subtask_symbfact(h)  # (the root's rows stay in their order)
    pastix.subtask_blend(h)
    pastix.set_amd_iparm(h, pastix.amd_iparm.profile, 1)
    pastix.task_numfact(h, S)
    assert pastix.kernel_times(h)["update_acc"][1] == launches * (2 if facto == F.LU else 1)
    pastix.finalize(h)
