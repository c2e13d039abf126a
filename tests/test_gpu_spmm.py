"""Near field of several right-hand sides in shared passes over the values
(k_spmm_cols) against the single-vector operator, column by column, where its
tilings change: leaves of at most 8, 16, 32, 64 and more rows, 8 and 16
right-hand sides per pass with a remainder, odd column counts.

Both paths sum each row in the same order; what differs from call to call is
the order of the far field's atomic adds: at most the rounding of a few
hundred terms, 1e-13 of the vector's norm in FP64 and 1e-6 in FP32.
"""
import numpy as np
import pytest

import pibem_amd as P
from pibem_amd import mesh as M

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("n,deg,leaf,rhs", [(10, 1, 8, (16, 17)), (13, 1, 20, (16, 33)), (12, 1, 48, (16,)),
                                            (11, 2, 96, (16, 19)), (16, 1, 400, (16,)), (40, 1, 96, (8, 9, 15))])
@pytest.mark.parametrize("precision", [P.PBFMM_FP64, P.PBFMM_MIXED])
def test_columns_equal_single_vector(n, deg, leaf, rhs, precision):
    from pibem_amd import hip
    pr = M.config_sphere(n, 4, deg)
    pr.max_nodes_per_leaf = leaf
    f = P.setup(pr, precision)
    bp = P.BEMProblem(f)
    bp.compute_alpha()
    N = f.n
    print(f"\n[case] sphere n={n} q{deg} N={N} leaf={leaf} precision={precision} {f.work_counts()}", flush=True)
    rng = np.random.default_rng(3)
    out = hip.DeviceArray(N)
    for R in rhs:
        x = rng.uniform(-1, 1, (R, N))
        x[1] = 0.0
        dx, dy = hip.DeviceArray.from_numpy(x.ravel()), hip.DeviceArray(R * N)
        bp.vmult_dev_multi(dx.value, dy.value, R, None, precision)
        hip.synchronize()
        y = dy.numpy().reshape(R, N)
        assert not y[1].any()
        tol = 1e-13 if precision == P.PBFMM_FP64 else 1e-6
        for r in (0, 2, R // 2, R - 1):
            v = hip.DeviceArray.from_numpy(x[r])
            bp.vmult_dev(v.value, out.value, precision)
            hip.synchronize()
            e = rel(y[r], out.numpy())
            print(f"  R={R} column {r}: {e:.1e}", flush=True)
            assert e <= tol
    f.close()


def test_nonfinite_column_stays_its_own():
    """An infinity in one right-hand side reaches no other one."""
    from pibem_amd import hip
    pr = M.config_sphere(12, 4)
    f = P.setup(pr)
    bp = P.BEMProblem(f)
    bp.compute_alpha()
    N, R = f.n, 16
    x = np.random.default_rng(4).uniform(-1, 1, (R, N))
    dx, dy = hip.DeviceArray.from_numpy(x.ravel()), hip.DeviceArray(R * N)
    bp.vmult_dev_multi(dx.value, dy.value, R)
    hip.synchronize()
    y0 = dy.numpy().reshape(R, N)
    x[5, 7] = np.inf
    dx.upload(x.ravel())
    bp.vmult_dev_multi(dx.value, dy.value, R)
    hip.synchronize()
    y1 = dy.numpy().reshape(R, N)
    keep = [r for r in range(R) if r != 5]
    assert np.isfinite(y1[keep]).all() and rel(y1[keep], y0[keep]) <= 1e-13 and not np.isfinite(y1[5]).all()
    f.close()
