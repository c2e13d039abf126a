"""A handle's first application of a precision inside a caller's capture, at
sizes whose launch plan keeps buffers (the M2L's slots, plans 5 and 92) or a
second stream (plan 24) that it makes on first use: the capture ends well, and
three replays, with eager applications between them, equal those.

The captured application may add with atomics where the eager ones use slots:
1e-13 of the vector's norm in FP64, 1e-6 in FP32, the rounding of a few
hundred terms.
"""
import ctypes as C

import numpy as np
import pytest

import pibem_amd as P
from pibem_amd import mesh as M

pytestmark = pytest.mark.gpu


def ok(rc):
    assert rc == 0, rc


@pytest.mark.parametrize("n,order,leaf,plan", [(64, 6, 20, None), (80, 4, 20, None), (80, 4, 128, None),
                                               (10, 4, 20, 4), (10, 4, 20, 24), (10, 4, 20, 92)])
@pytest.mark.parametrize("precision", [P.PBFMM_FP64, P.PBFMM_MIXED])
def test_first_application_captured(n, order, leaf, plan, precision):
    from pibem_amd import hip
    rt = hip.hip()
    pr = M.config_sphere(n, order)
    stream, graph, run = C.c_void_p(), C.c_void_p(), C.c_void_p()
    ok(rt.hipStreamCreate(C.byref(stream)))
    f = P.BEMFMA(trunc_order=order, num_octree_levels=pr.levels, max_nodes_per_leaf=leaf, quad_order=pr.quad_order,
                 sing_quad_order=pr.sing_quad_order, stream=stream.value, precision=P.PBFMM_MIXED)
    f.init_fma(pr.mesh, pr.dirichlet)
    f.generate_octree_blocking()
    f.direct_integrals()
    f.multipole_integrals()
    bp = P.BEMProblem(f)
    bp.compute_alpha()
    if plan is not None:
        f.set_side_fusion(precision, plan)
    print(f"\n[case] sphere N={f.n} order {order} leaf {leaf} plan {plan} precision {precision}", flush=True)
    src = np.random.default_rng(9).uniform(-1, 1, f.n)
    x, y = hip.DeviceArray.from_numpy(src), hip.DeviceArray(f.n)
    hip.synchronize()
    ok(rt.hipStreamBeginCapture(stream, C.c_int(1)))  # thread-local mode
    bp.vmult_dev(x.value, y.value, precision)
    ok(rt.hipStreamEndCapture(stream, C.byref(graph)))
    ok(rt.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)))
    for k in range(3):
        x.upload(src * 0.5 ** k)
        y.upload(np.zeros(f.n))
        hip.synchronize()
        ok(rt.hipGraphLaunch(run, stream))
        hip.synchronize()
        got = y.numpy()
        bp.vmult_dev(x.value, y.value, precision)
        hip.synchronize()
        e = np.linalg.norm(got - y.numpy()) / np.linalg.norm(got)
        print(f"  replay {k}: {e:.1e}", flush=True)
        assert e <= (1e-13 if precision == P.PBFMM_FP64 else 1e-6)
    ok(rt.hipGraphExecDestroy(run))
    ok(rt.hipGraphDestroy(graph))
    f.close()
    ok(rt.hipStreamDestroy(stream))
