"""The launch plan that the sizes suggest for a new handle's first
applications against plan 0, on either side of the rule's lines: few values
with and without M2P work, many M2L pairs, many values.

A plan changes where and when the far field's parts run, so the two differ by
the order of atomic adds and of the two streams' sums: at most the rounding
of a few hundred terms, 1e-13 of the vector's norm in FP64, 1e-6 in FP32.
"""
import numpy as np
import pytest

import pibem_amd as P
from pibem_amd import mesh as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,order,leaf", [(10, 4, 20), (16, 4, 20), (32, 6, 64), (64, 6, 20), (64, 6, 96),
                                          (80, 4, 20), (80, 4, 128)])
def test_first_applications_equal_plan_0(n, order, leaf):
    from pibem_amd import hip
    pr = M.config_sphere(n, order)
    pr.max_nodes_per_leaf = leaf
    f = P.setup(pr, P.PBFMM_MIXED)
    bp = P.BEMProblem(f)
    bp.compute_alpha()
    print(f"\n[case] sphere n={n} N={f.n} order={order} leaf={leaf} {f.work_counts()}", flush=True)
    dx = hip.DeviceArray.from_numpy(np.random.default_rng(5).uniform(-1, 1, f.n))
    dy = hip.DeviceArray(f.n)
    for precision, name, tol in ((0, "fp64", 1e-13), (1, "fp32", 1e-6)):
        got = []
        for plan in (None, 0):
            if plan is not None:
                f.set_side_fusion(precision, plan)
            for _ in range(2):
                bp.vmult_dev(dx.value, dy.value, precision)
                hip.synchronize()
                got.append(dy.numpy())
            if plan is None:
                assert f.tuning_state()[f"side_fusion_{name}"] == -1
        for y in got[:3]:
            e = np.linalg.norm(y - got[3]) / np.linalg.norm(got[3])
            print(f"  {name}: {e:.1e}", flush=True)
            assert e <= tol
    f.close()
