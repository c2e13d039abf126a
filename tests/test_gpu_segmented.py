"""Lockstep solves against one solve per right-hand side where the segmented
Arnoldi kernels' tilings change: parts within one chunk of 2048 rows, of a
chunk and a remainder, and of several chunks, with 2, 3 and 5 parts (chunks
are cut at part ends, workgroups of 256 rows at chunk ends).

Both solves reach a relative residual of 1e-10; the operator's condition
number is below 100 here, so the solutions agree to 2e-8.
"""
import numpy as np
import pytest

import pibem_amd as P
from pibem_amd import mesh as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,rhs", [(6, 2), (10, 3), (18, 2), (20, 5), (40, 3)])
@pytest.mark.parametrize("restart", [7, 100])
def test_lockstep_equals_single(n, rhs, restart):
    from pibem_amd import hip
    pr = M.config_sphere(n, 4)
    f = P.setup(pr)
    bp = P.BEMProblem(f)
    bp.compute_alpha()
    bp.fma_preconditioner()
    N = f.n
    print(f"\n[case] sphere N={N} rhs={rhs} restart={restart}", flush=True)
    b = np.random.default_rng(n).uniform(-1, 1, (rhs, N))
    db, dx = hip.DeviceArray.from_numpy(b.ravel()), hip.DeviceArray.from_numpy(np.zeros(rhs * N))
    f.gmres_dev_multi(db.value, dx.value, rhs, N, 1e-10, restart, 2000, P.PBFMM_FP64)
    hip.synchronize()
    x = dx.numpy().reshape(rhs, N)
    for r in range(rhs):
        d1, d2 = hip.DeviceArray.from_numpy(b[r]), hip.DeviceArray.from_numpy(np.zeros(N))
        f.gmres_dev(d1.value, d2.value, 1e-10, restart, 2000, P.PBFMM_FP64)
        hip.synchronize()
        y = d2.numpy()
        e = np.linalg.norm(x[r] - y) / np.linalg.norm(y)
        print(f"  rhs {r}: {e:.1e}", flush=True)
        assert e <= 2e-8
    f.close()


@pytest.mark.parametrize("restart", [9, 300])
def test_batch_equals_single(restart):
    """Uneven parts as one batch, whose restart has no upper limit."""
    from pibem_amd import hip
    problems = [M.config_sphere(n, 4) for n in (6, 20, 10)]
    batch = P.setup_batch(problems)
    b = np.random.default_rng(1).uniform(-1, 1, batch.n)
    db, dx = hip.DeviceArray.from_numpy(b), hip.DeviceArray.from_numpy(np.zeros(batch.n))
    batch.gmres_batch_dev(db.value, dx.value, 1e-10, restart, 2000, P.PBFMM_FP64)
    hip.synchronize()
    x, at = dx.numpy(), 0
    for pr in problems:
        f = P.setup(pr)
        P.BEMProblem(f).compute_alpha()
        d1, d2 = hip.DeviceArray.from_numpy(b[at:at + f.n]), hip.DeviceArray.from_numpy(np.zeros(f.n))
        f.gmres_dev(d1.value, d2.value, 1e-10, 100, 2000, P.PBFMM_FP64)
        hip.synchronize()
        y = d2.numpy()
        assert np.linalg.norm(x[at:at + f.n] - y) <= 2e-8 * np.linalg.norm(y)
        at += f.n
        f.close()
    batch.close()
