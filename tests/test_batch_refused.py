"""A batch that is refused (not the analysed one) leaves the instance as it
was: the same call is refused again, the analysed batch is still accepted, and
its factor can still be used.  Reference: numpy's norms, dense solves."""
import numpy as np
import pytest
import scipy.sparse as sps

from pastix_amd import pastix, spm

F = pastix.factotype
KS = [3, 4, 7]


def _analysed():
    mats = [spm.laplacian5_2d(k) + 0.5 * sps.eye(k * k) for k in KS]
    S = [spm.Spm(A, symmetric=True) for A in mats]
    ip, dp = pastix.initParam()
    ip[pastix.iparm.factorization] = F.LLT
    h = pastix.init(ip, dp)
    pastix.batch_analyze(h, S, None)
    # the same systems with fewer entries in the last one, with another order
    # of two, with one left out of the symmetric storage
    fewer = S[:2] + [spm.Spm(sps.csc_matrix(2.0 * sps.eye(49)), symmetric=True)]
    swapped = [S[1], S[0], S[2]]
    general = [spm.Spm(A, symmetric=False) for A in mats]
    return h, mats, S, (fewer, swapped, general)


def _refused(h, S):
    with pytest.raises(pastix.PastixError, match="returned 7"):
        pastix.batch_numfact(h, S)


def _accepted(h, S):
    """True when the batch passes the comparison (without a GPU the engine's
    set-up fails after it)."""
    h.dparm[pastix.dparm.a_norm] = -1.0
    try:
        pastix.batch_numfact(h, S)
    except pastix.PastixError as e:
        assert "returned 7" not in str(e)
    return float(h.dparm[pastix.dparm.a_norm]) > 0.0


@pytest.mark.parametrize("calls", ["gbg", "bg", "gbbg", "bbg", "gbgbg"])
@pytest.mark.parametrize("which", [0, 1, 2])
def test_refused_batch_changes_nothing(calls, which):
    h, mats, S, bad = _analysed()
    # the threshold's norm: the smallest of the systems' own
    ref = min(np.linalg.norm(A.toarray()) for A in mats)
    for c in calls:
        if c == "b":
            _refused(h, bad[which])
        else:
            assert _accepted(h, S)
            assert abs(float(h.dparm[pastix.dparm.a_norm]) - ref) <= 1e-13 * ref
    pastix.finalize(h)


@pytest.mark.gpu
@pytest.mark.parametrize("which", [0, 1, 2])
def test_factor_after_a_refused_batch(which):
    h, mats, S, bad = _analysed()
    rng = np.random.default_rng(which)
    bs = [rng.uniform(-1.0, 1.0, (k * k, 2)) for k in KS]

    def solved():
        for A, b, x in zip(mats, bs, pastix.batch_solve(h, bs)):
            xd = np.linalg.solve(A.toarray(), b)
            assert np.abs(x - xd).max() <= 1e-11 * np.abs(xd).max()

    pastix.batch_numfact(h, S)
    solved()
    _refused(h, bad[which])
    _refused(h, bad[which])
    solved()
    pastix.batch_numfact(h, S)
    solved()
    pastix.finalize(h)
