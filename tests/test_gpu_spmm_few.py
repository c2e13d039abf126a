"""Two to seven right-hand sides in shared passes over the near field, which
they take from 256 MB of values on (two of them from 1 GB), against the
single-vector operator, column by column; and two on 256 MB, which stay apart.

Both paths sum each row in the same order; what differs from call to call is
the order of the far field's atomic adds: at most the rounding of a few
hundred terms, 1e-13 of the vector's norm in FP64 and 1e-6 in FP32.
"""
import numpy as np
import pytest

import pibem_amd as P
from pibem_amd import mesh as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,leaf,rhs,precision,megabytes", [
    (80, 128, (2, 3, 5, 7), P.PBFMM_FP64, 256), (64, 1600, (2, 3), P.PBFMM_FP64, 1024),
    (64, 1600, (2, 3, 7), P.PBFMM_MIXED, 256), (64, 6200, (2, 4), P.PBFMM_MIXED, 1024)])
def test_columns_equal_single_vector(n, leaf, rhs, precision, megabytes):
    from pibem_amd import hip
    pr = M.config_sphere(n, 4)
    pr.max_nodes_per_leaf = leaf
    f = P.setup(pr, precision)
    bp = P.BEMProblem(f)
    bp.compute_alpha()
    N = f.n
    w = f.work_counts()
    mb = w["near_values"] * (8 if precision == P.PBFMM_FP64 else 4) / 2 ** 20
    print(f"\n[case] sphere n={n} N={N} leaf={leaf} precision={precision} leaves {w['leaves']}, {mb:.0f} MB", flush=True)
    assert mb >= megabytes
    rng = np.random.default_rng(3)
    out = hip.DeviceArray(N)
    tol = 1e-13 if precision == P.PBFMM_FP64 else 1e-6
    for R in rhs:
        x = rng.uniform(-1, 1, (R, N))
        dx, dy = hip.DeviceArray.from_numpy(x.ravel()), hip.DeviceArray(R * N)
        bp.vmult_dev_multi(dx.value, dy.value, R, None, precision)
        hip.synchronize()
        y = dy.numpy().reshape(R, N)
        for r in range(R):
            v = hip.DeviceArray.from_numpy(x[r])
            bp.vmult_dev(v.value, out.value, precision)
            hip.synchronize()
            e = np.linalg.norm(y[r] - out.numpy()) / np.linalg.norm(y[r])
            print(f"  R={R} column {r}: {e:.1e}", flush=True)
            assert e <= tol
    f.close()
