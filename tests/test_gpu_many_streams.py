"""Handles enough that their streams share hardware queues (a process has
four): whichever second stream each one took, the operator with the SpMV on it
(plan 24) equals plan 0, with all handles' applications in flight at once.
The bars are those of the other plan tests: 1e-13 of the norm in FP64."""
import numpy as np
import pytest

import pibem_amd as P
from pibem_amd import hip
from pibem_amd import mesh as M

pytestmark = pytest.mark.gpu


def test_second_streams_of_many_handles():
    pr = M.config_sphere(64, 4)
    pr.max_nodes_per_leaf = 96
    fs = [P.setup(pr) for _ in range(6)]
    assert fs[0].work_counts()["near_values"] >= 8000000
    bps = [P.BEMProblem(f) for f in fs]
    rng = np.random.default_rng(4)
    xs = [hip.DeviceArray.from_numpy(rng.uniform(-1, 1, f.n)) for f in fs]
    ys = [hip.DeviceArray(f.n) for f in fs]
    got = {}
    for bp in bps:
        bp.compute_alpha()
    for plan in (0, 24):
        for f in fs:
            f.set_side_fusion(P.PBFMM_FP64, plan)
        for _ in range(5):
            for bp, x, y in zip(bps, xs, ys):
                bp.vmult_dev(x.value, y.value, P.PBFMM_FP64)
        hip.synchronize()
        got[plan] = [y.numpy() for y in ys]
    for k in range(len(fs)):
        e = np.linalg.norm(got[24][k] - got[0][k]) / np.linalg.norm(got[0][k])
        print(f"  handle {k}: {e:.1e}", flush=True)
        assert e <= 1e-13
    for f in fs:
        f.close()
