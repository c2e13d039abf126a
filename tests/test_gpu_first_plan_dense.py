"""The launch plan that the sizes suggest where each M2L pair has a thousand
near-field values or more, on either side of that line, against plan 0: large
leaves, and a mirrored hull.

A plan changes where and when the far field's parts run, so the two differ by
the order of atomic adds and of the two streams' sums: at most the rounding
of a few hundred terms, 1e-13 of the vector's norm in FP64, 1e-6 in FP32.
"""
import numpy as np
import pytest

import pibem_amd as P
from pibem_amd import mesh as M

pytestmark = pytest.mark.gpu


def sphere(n, order, leaf):
    pr = M.config_sphere(n, order)
    pr.max_nodes_per_leaf = leaf
    return pr


def half_hull(nx, nz, order, leaf):
    pr = M.config_wigley_half(nx, nz, order)
    pr.max_nodes_per_leaf = leaf
    return pr


CASES = [("sphere leaf 96", lambda: sphere(64, 6, 96), False), ("sphere leaf 128", lambda: sphere(80, 4, 128), None),
         ("sphere leaf 200", lambda: sphere(64, 5, 200), True), ("half hull", lambda: half_hull(240, 30, 4, 64), None)]


@pytest.mark.parametrize("name,make,dense", CASES, ids=[c[0] for c in CASES])
def test_first_applications_equal_plan_0(name, make, dense):
    from pibem_amd import hip
    f = P.setup(make(), P.PBFMM_MIXED)
    bp = P.BEMProblem(f)
    bp.compute_alpha()
    w = f.work_counts()
    print(f"\n[case] {name} N={f.n} values {w['near_values']} pairs {w['m2l_pairs']}", flush=True)
    if dense is not None:
        assert w["near_values"] >= 8000000 and (w["near_values"] >= 1000 * w["m2l_pairs"]) == dense
    x = hip.DeviceArray.from_numpy(np.random.default_rng(7).uniform(-1, 1, f.n))
    y = hip.DeviceArray(f.n)
    for precision, tol in ((0, 1e-13), (1, 1e-6)):
        got = []
        for plan in (None, 0):
            if plan is not None:
                f.set_side_fusion(precision, plan)
            for _ in range(2):
                bp.vmult_dev(x.value, y.value, precision)
                hip.synchronize()
                got.append(y.numpy())
        for v in got[:3]:
            e = np.linalg.norm(v - got[3]) / np.linalg.norm(got[3])
            print(f"  precision {precision}: {e:.1e}", flush=True)
            assert e <= tol
    f.close()
