"""The leaf-size autotuner compares leaf sizes as a handle in long use runs
them: every handle that it times has chosen its launch plans and its graph
before the timed solves."""
import pytest

import pibem_amd as P
from pibem_amd import mesh as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [P.PBFMM_FP64, P.PBFMM_MIXED])
def test_timed_solves_run_timed_plans(precision, monkeypatch):
    seen = []
    solve = P.BEMFMA.gmres_dev

    def watched(self, *args, **kwargs):
        before = self.tuning_state()
        out = solve(self, *args, **kwargs)
        seen.append((self, before))
        return out

    monkeypatch.setattr(P.BEMFMA, "gmres_dev", watched)
    pr = M.config_sphere(12, 4)
    best, times, info, _ = P.tune_leaf_size(pr, precision, solves=2, start=20, ladder=(12, 20, 32))
    assert set(times) == {12, 20, 32} and len(seen) == 9
    name = "fp32" if precision == P.PBFMM_MIXED else "fp64"
    for k in range(3):
        for _, before in seen[3 * k + 1:3 * k + 3]:  # the solves after the warm-up one
            assert before["side_fusion_" + name] >= 0 and before["graph_" + name] >= 0, before
