"""A call that fails for memory leaves its handle, and others, usable: buffers
that it dropped are made again by the next call, and the runtime's error is
not reported a second time.  (A batch's restart length has no upper limit, so
its basis can be asked to exceed any memory.)"""
import numpy as np
import pytest

import pibem_amd as P
from pibem_amd import hip
from pibem_amd import mesh as M

pytestmark = pytest.mark.gpu


def test_batch_after_a_basis_that_does_not_fit():
    batch = P.setup_batch([M.config_sphere(n, 4) for n in (6, 10)])
    other = P.setup(M.config_sphere(8, 4))
    bp = P.BEMProblem(other)
    bp.compute_alpha()
    x = np.random.default_rng(2).uniform(-1, 1, other.n)
    y = bp.vmult(x)
    b = hip.DeviceArray.from_numpy(np.random.default_rng(1).uniform(-1, 1, batch.n))
    s = hip.DeviceArray.from_numpy(np.zeros(batch.n))
    batch.gmres_batch_dev(b.value, s.value, 1e-8, 20, 500, P.PBFMM_FP64)
    want = s.numpy()
    with pytest.raises(P.PbfmmError, match="out of memory"):
        batch.gmres_batch_dev(b.value, s.value, 1e-8, 10 ** 9, 500, P.PBFMM_FP64)
    assert np.linalg.norm(bp.vmult(x) - y) <= 1e-13 * np.linalg.norm(y)
    s.upload(np.zeros(batch.n))
    hip.synchronize()
    batch.gmres_batch_dev(b.value, s.value, 1e-8, 20, 500, P.PBFMM_FP64)
    assert np.linalg.norm(s.numpy() - want) <= 1e-10 * np.linalg.norm(want)
    batch.close()
    other.close()
