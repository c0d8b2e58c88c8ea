"""New values of matrices with full rows among short ones (the chunks whose
sums make up the norm end at rows, entries and systems), no GPU: the norm
within 1e-13 of numpy's, in one instance and as the smallest of a batch's."""
import numpy as np
import pytest
import scipy.sparse as sps

from pastix_amd import pastix, spm

F = pastix.factotype


def _matrix(n, full, seed):
    rng = np.random.default_rng(seed)
    A = sps.diags([np.full(n, 4.0 + seed), np.full(n - 1, -1.0), np.full(n - 1, -1.0)], [0, 1, -1]).tolil()
    for r in full:
        A[r, :] = rng.uniform(0.1, 1.0, n)
    A = sps.csc_matrix(A)
    A = sps.csc_matrix(sps.tril(A) + sps.tril(A, -1).T)
    A[full, full] = 2.0 * n
    return sps.csc_matrix(A)


CASES = [(700, []), (700, [0]), (1200, [3, 4, 5, 600, 1199]), (1500, list(range(1500)))]


@pytest.mark.parametrize("symmetric", [True, False])
@pytest.mark.parametrize("n,full", CASES)
def test_norm(n, full, symmetric):
    A = _matrix(n, full, 1)
    S = spm.Spm(A.copy(), symmetric=symmetric)
    norm = sps.linalg.norm(A)
    ip, dp = pastix.initParam()
    ip[pastix.iparm.factorization] = F.LLT if symmetric else F.LU
    h = pastix.init(ip, dp)
    pastix.task_analyze(h, S)
    for scale in (1.0, 0.5, 3.0):
        S.set_values(sps.csc_matrix(scale * A))
        pastix.subtask_spm2bcsc(h, S)
        ref = scale * norm
        assert abs(float(h.dparm[pastix.dparm.a_norm]) - ref) <= 1e-13 * ref
    pastix.finalize(h)


def test_smallest_norm_of_a_batch():
    mats = [_matrix(n, full, 1 + k) for k, (n, full) in enumerate(CASES)]
    S = [spm.Spm(A, symmetric=True) for A in mats]
    ip, dp = pastix.initParam()
    ip[pastix.iparm.factorization] = F.LLT
    h = pastix.init(ip, dp)
    pastix.batch_analyze(h, S, None)
    for scales in ((1, 1, 1, 1), (900, 1, 1, 1), (900, 900, 0.01, 1), (900, 900, 900, 1e-3)):
        for s, A, f in zip(S, mats, scales):
            s.set_values(sps.csc_matrix(f * A))
        try:
            pastix.batch_numfact(h, S)
        except pastix.PastixError:
            pass  # without a GPU the engine's set-up fails, after the norms
        ref = min(f * sps.linalg.norm(A) for A, f in zip(mats, scales))
        assert abs(float(h.dparm[pastix.dparm.a_norm]) - ref) <= 1e-13 * ref
    pastix.finalize(h)
