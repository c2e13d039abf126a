"""M2L on one workgroup per compute unit beside the SpMV, on either side of
the lines that choose it (near-field values per M2L pair, by precision and by
the translations' workgroup size): narrow (order 6) and wide (orders 5, 8, 10)
workgroups, 317 and 452 values per pair.

Plan 24 forks the SpMV and plan 0 does not; the two differ by the order of
atomic adds, at most the rounding of a few hundred terms: 1e-13 of the
vector's norm in FP64, 1e-6 in FP32.
"""
import numpy as np
import pytest

import pibem_amd as P
from pibem_amd import mesh as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,leaf", [(5, 48), (5, 96), (6, 48), (6, 96), (8, 96), (6, 200), (10, 200)])
def test_plan_24_equals_plan_0(order, leaf):
    from pibem_amd import hip
    m = M.cube_sphere(64, 1, (1.0, 1.0, 1.0), equiangular=True)
    f = P.BEMFMA(trunc_order=order, max_nodes_per_leaf=leaf, precision=P.PBFMM_MIXED)
    f.init_fma(m, M.dirichlet_mask(m, M.cell_centroids(m)[:, 2] > 0))
    f.generate_octree_blocking()
    f.direct_integrals()
    f.multipole_integrals()
    w = f.work_counts()
    per_pair = w["near_values"] / w["m2l_pairs"]
    print(f"\n[case] sphere N={f.n} order {order} leaf {leaf}: {per_pair:.0f} values per pair", flush=True)
    bp = P.BEMProblem(f)
    bp.compute_alpha()
    dx = hip.DeviceArray.from_numpy(np.random.default_rng(5).uniform(-1, 1, f.n))
    dy = hip.DeviceArray(f.n)
    for precision, tol in ((P.PBFMM_FP64, 1e-13), (P.PBFMM_MIXED, 1e-6)):
        got = []
        for plan in (0, 24, 24):
            f.set_side_fusion(precision, plan)
            bp.vmult_dev(dx.value, dy.value, precision)
            hip.synchronize()
            got.append(dy.numpy())
        e = [np.linalg.norm(y - got[0]) / np.linalg.norm(got[0]) for y in got[1:]]
        print(f"  precision {precision}: {e[0]:.1e} {e[1]:.1e}", flush=True)
        assert max(e) <= tol
    f.close()
