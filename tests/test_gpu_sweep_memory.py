"""Device memory of the solve sweeps: the vectors of 64 right-hand sides where
they are small, else of 32 until a call of more, none beyond a server's budget,
and the results before and after they are replaced."""
import numpy as np
import pytest

from pastix_amd import pastix, spm
from tests.helpers import analyse

pytestmark = pytest.mark.gpu
F = pastix.factotype
SMALL, LARGE = (13, 12, 11), (66, 65, 64)


def _berr(A, x, b):
    return max(float(np.abs(b[:, c] - A @ x[:, c]).max() / (abs(A).sum(axis=1).max() * np.abs(x[:, c]).max() +
                                                            np.abs(b[:, c]).max())) for c in range(b.shape[1]))


@pytest.mark.parametrize("prec", [spm.SpmDouble, spm.SpmFloat])
@pytest.mark.parametrize("facto,grid", [(F.LLT, SMALL), (F.LU, SMALL), (F.LLT, LARGE)])
def test_first_call_of_many(facto, grid, prec):
    A = spm.laplacian7(*grid, diag=6.0) if facto == F.LLT else spm.convection_diffusion27(*grid, seed=3)
    n, fsz = A.shape[0], 8 if prec == spm.SpmDouble else 4
    big = {"min_bs": 16, "max_bs": 40} if grid == SMALL else {}
    h, S, _ = analyse(A, facto == F.LLT, facto, grid=grid, **big)
    pastix.set_amd_iparm(h, pastix.amd_iparm.factor_precision, prec)
    pastix.task_numfact(h, S)

    def solve(nrhs):
        _, b = spm.rhs_from_x(A, nrhs, seed=nrhs)
        x = b.copy(order="F")
        pastix.task_solve(h, S, x)
        assert _berr(A, x, b) <= (1e-14 if prec == spm.SpmDouble else 1e-6), nrhs
        return pastix.device_bytes(h)

    base = solve(1)
    assert solve(32) == base + 31 * n * fsz   # the permuted right-hand sides
    wide = solve(33)
    if grid == SMALL:
        assert wide == base + 32 * n * fsz
    else:
        # 32 more columns of the sweep, more than 256 MiB
        assert wide - base > 32 * n * fsz + (256 << 20)
    assert solve(64) == wide + 31 * n * fsz
    assert solve(1) == wide + 31 * n * fsz
    assert solve(70) == wide + 37 * n * fsz
    pastix.finalize(h)


def test_interface_sweep_of_many():
    """The Schur rows' update-buffer entries read as zero in the wider buffer
    too: 40 columns at once as 20 and 20."""
    grid = (9, 8, 7)
    A = spm.laplacian7(*grid, coef=(1.0, 1.0, 0.3))
    n = A.shape[0]
    got = []
    for parts in ((40,), (20, 20)):
        S = spm.Spm(A, symmetric=True)
        ip, dp = pastix.initParam()
        ip[pastix.iparm.factorization] = F.LLT
        ip[pastix.iparm.min_blocksize] = 16
        ip[pastix.iparm.max_blocksize] = 32
        h = pastix.init(ip, dp)
        pastix.setSchurUnknownList(h, np.arange(n // 3, dtype=np.int64))
        ip[pastix.iparm.schur_solv_mode] = pastix.solv_mode.Interface
        pastix.task_analyze(h, S)
        pastix.task_numfact(h, S)
        _, b = spm.rhs_from_x(A, 40, seed=8)
        out, c0 = [], 0
        for p in parts:
            x = np.asfortranarray(b[:, c0:c0 + p].copy())
            pastix.subtask_applyorder(h, pastix.dir.Forward, x)
            pastix.subtask_trsm(h, pastix.side.Left, pastix.uplo.Lower, pastix.trans.NoTrans, pastix.diag.NonUnit, x)
            out.append(x)
            c0 += p
        got.append(np.hstack(out))
        pastix.finalize(h)
    assert np.abs(got[0] - got[1]).max() <= 1e-13 * np.abs(got[1]).max()


@pytest.mark.parametrize("grid,percentage,max_rhs,wider", [(LARGE, 95, 64, True), (LARGE, 95, 32, False),
                                                            (LARGE, 100, 64, False), (SMALL, 95, 64, False)])
def test_server(grid, percentage, max_rhs, wider):
    """A server's slots take the wider sweeps at its creation, from the memory
    its budget leaves free, or not at all."""
    A = spm.laplacian7(*grid, coef=(1.0, 1.0, 0.01))
    n = A.shape[0]
    S = spm.Spm(A, symmetric=True)
    ip, dp = pastix.initParam()
    ip[pastix.iparm.factorization] = F.LLT
    ip[pastix.iparm.refinement] = pastix.refine.CG
    ip[pastix.iparm.gpu_memory_percentage] = percentage
    ip[pastix.iparm.ordering] = pastix.order.Personal
    h = pastix.init(ip, dp)
    pastix.set_amd_iparm(h, pastix.amd_iparm.factor_precision, spm.SpmFloat)
    pastix.set_amd_iparm(h, pastix.amd_iparm.resident_input, 1)
    o = pastix.orderGrid(*grid)
    h.order = o
    pastix.subtask_order(h, S, o)
    pastix.subtask_symbfact(h)
    pastix.subtask_reordering(h)
    pastix.subtask_blend(h)
    pastix.task_numfact(h, S)
    before = pastix.device_bytes(h)
    srv = pastix.Server([h], max_rhs=max_rhs)
    created = pastix.device_bytes(h)
    assert (created > before) == wider
    rng = np.random.default_rng(2)
    for nrhs in (1, max_rhs):
        b = rng.uniform(-1.0, 1.0, (n, nrhs))
        x, _, _ = srv.wait(srv.submit_solve(b.copy(order="F")))
        assert _berr(A, x, b) <= 1e-12
    held = srv.memory()["held"]
    # the admitted blocks and a few words per row for the segmented sums
    assert pastix.device_bytes(h) - created <= held + 16 * n + 4096
    srv.close()
    pastix.finalize(h)
