"""The one-pass update for levels of narrow sources does not depend on how
large the target's panel is (host analysis only, no GPU)."""
import ctypes as ct

import numpy as np
import pytest
import scipy.sparse as sps

from pastix_amd import pastix, spm


def _arrow(root, leaves):
    """`leaves` single columns, each with entries in three rows of a dense
    block of `root` columns (filled by its first one, which couples to all)."""
    n = leaves + root
    r, c = [np.arange(n)], [np.arange(n)]
    for k in range(leaves):
        r.append(leaves + np.array([1, 2, 3]) + k % 7)
        c.append(np.full(3, k))
    r.append(leaves + np.arange(1, root))
    c.append(np.full(root - 1, leaves))
    r, c = np.concatenate(r), np.concatenate(c)
    L = sps.coo_matrix((np.where(r == c, 100.0, 1.0), (r, c)), shape=(n, n))
    return sps.csc_matrix(L + sps.tril(L, -1).T)


@pytest.mark.parametrize("root", [300, 16500])
def test_narrow_sources_of_a_wide_target(root):
    leaves = 60
    A = _arrow(root, leaves)
    n = A.shape[0]
    S = spm.Spm(A, symmetric=True)
    ip, dp = pastix.initParam()
    ip[pastix.iparm.factorization] = pastix.factotype.LLT
    ip[pastix.iparm.ordering] = pastix.order.Personal
    ip[pastix.iparm.min_blocksize] = 16
    ip[pastix.iparm.max_blocksize] = 20000
    h = pastix.init(ip, dp)
    # the given order: every leaf a supernode, the root the last one
    tabs = [np.arange(n), np.arange(n), np.append(np.arange(leaves + 1), n), np.append(np.full(leaves, leaves), -1)]
    tabs = [np.ascontiguousarray(t, dtype=np.int64) for t in tabs]
    o = pastix.pastix_order_t()
    o.vertnbr, o.cblknbr = n, leaves + 1
    o.permtab, o.peritab, o.rangtab, o.treetab = [t.ctypes.data_as(ct.POINTER(ct.c_int64)) for t in tabs]
    pastix.subtask_order(h, S, o)
    pastix.subtask_symbfact(h)
    pastix.subtask_reordering(h)
    pastix.subtask_blend(h)
    assert np.diff(pastix.symbol(h)["cblk_fcol"]).max() == root
    # 60 sources of one column into one tile, in one pass; the root updates nothing
    assert pastix.level_info(h)[:, :3].tolist() == [[leaves, 1, 1], [1, 0, 0]]
    pastix.finalize(h)
