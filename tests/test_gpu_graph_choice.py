"""The unasked choice between direct steps and graph replays: it is made on a
solve's own steps, half of them replays, and replayed steps count towards the
timing of the launch plans as direct ones do.

Solves to 1e-8 are compared with the bars of the graph tests: 1e-10 (FP64),
1e-7 (mixed).
"""
import numpy as np
import pytest

import pibem_amd as P
from pibem_amd import hip
from pibem_amd import mesh as M

pytestmark = pytest.mark.gpu


def make():
    pr = M.config_sphere(16, 5)
    f = P.setup(pr, P.PBFMM_MIXED)
    bp = P.BEMProblem(f)
    return f, hip.DeviceArray.from_numpy(bp.compute_rhs(pr.tmp_rhs))


def solve(f, rhs, precision):
    x = hip.DeviceArray(f.n)
    its, rr = f.gmres_dev(rhs.value, x.value, 1e-8, 100, 2000, precision)
    hip.synchronize()
    assert rr <= 1e-8
    return x.numpy(), its


@pytest.mark.parametrize("precision,name,bar", [(P.PBFMM_FP64, "fp64", 1e-10), (P.PBFMM_MIXED, "fp32", 1e-7)])
def test_choice_on_a_solves_steps(precision, name, bar):
    f, rhs = make()
    f.set_mixed_scheme(2)  # refinement: its inner solves take FP32 steps only
    print(f"\n[case] sphere N={f.n} {name}", flush=True)
    f.set_graph_mode(0)
    want, its0 = solve(f, rhs, precision)
    f.set_graph_mode(-1)
    for k in range(12):
        x, its = solve(f, rhs, precision)
        e = np.linalg.norm(x - want) / np.linalg.norm(want)
        st = f.tuning_state()
        print(f"  solve {k}: {its} steps ({its0}), graph {st['graph_' + name]}, {e:.1e}", flush=True)
        assert e <= bar and abs(its - its0) <= 2
    assert st["graph_" + name] in (0, 1)
    t = f.graph_timings()
    assert min(t[:2] if name == "fp64" else t[2:]) > 0
    f.close()


def test_replayed_steps_count_for_the_plans():
    f, rhs = make()
    print(f"\n[case] sphere N={f.n}, replays", flush=True)
    f.set_graph_mode(1)
    steps = 0
    while steps < 1100:
        steps += solve(f, rhs, P.PBFMM_FP64)[1]
    assert f.tuning_state()["side_fusion_fp64"] >= 0
    f.close()
