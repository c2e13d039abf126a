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


def test_capture_where_the_plan_would_be_timed():
    """An application among those that time the plans (the 9th to the 43rd),
    inside a caller's capture: it is not timed and replays; the eager ones
    after it go on and choose a plan."""
    import ctypes as C
    from pibem_amd import hip
    rt = hip.hip()

    def ok(rc):
        assert rc == 0, rc

    pr = M.config_sphere(16, 4)
    stream, graph, run = C.c_void_p(), C.c_void_p(), C.c_void_p()
    ok(rt.hipStreamCreate(C.byref(stream)))
    f = P.BEMFMA(trunc_order=pr.p, num_octree_levels=pr.levels, max_nodes_per_leaf=pr.max_nodes_per_leaf,
                 quad_order=pr.quad_order, sing_quad_order=pr.sing_quad_order, stream=stream.value)
    f.init_fma(pr.mesh, pr.dirichlet)
    f.generate_octree_blocking()
    f.direct_integrals()
    f.multipole_integrals()
    bp = P.BEMProblem(f)
    bp.compute_alpha()
    src = np.linspace(-1, 1, f.n)
    x, y = hip.DeviceArray.from_numpy(src), hip.DeviceArray(f.n)
    for _ in range(20):
        bp.vmult_dev(x.value, y.value, P.PBFMM_FP64)
    hip.synchronize()
    ok(rt.hipStreamBeginCapture(stream, C.c_int(1)))  # thread-local mode
    bp.vmult_dev(x.value, y.value, P.PBFMM_FP64)
    ok(rt.hipStreamEndCapture(stream, C.byref(graph)))
    ok(rt.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)))
    assert f.tuning_state()["side_fusion_fp64"] == -1
    for k in range(3):
        x.upload(src * 0.5 ** k)
        y.upload(np.zeros(f.n))
        hip.synchronize()
        ok(rt.hipGraphLaunch(run, stream))
        hip.synchronize()
        got = y.numpy()
        bp.vmult_dev(x.value, y.value, P.PBFMM_FP64)
        hip.synchronize()
        assert np.linalg.norm(got - y.numpy()) <= 1e-13 * np.linalg.norm(got), k
    for _ in range(30):
        bp.vmult_dev(x.value, y.value, P.PBFMM_FP64)
        hip.synchronize()
        assert np.linalg.norm(got - y.numpy()) <= 1e-13 * np.linalg.norm(got)
    assert f.tuning_state()["side_fusion_fp64"] >= 0
    ok(rt.hipGraphExecDestroy(run))
    ok(rt.hipGraphDestroy(graph))
    f.close()
    ok(rt.hipStreamDestroy(stream))
