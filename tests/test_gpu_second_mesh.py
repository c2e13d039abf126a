"""A handle that takes another mesh (pbfmm_init_fma again) does on it what a
new handle does: every buffer, plan and timed choice that the first mesh left
goes with it, whatever was run on it (single applications up to a timed plan,
solves in both precisions, right-hand sides in lockstep, slots of the M2L,
graphs, projections), and what the caller chose stays.

FP64 results differ by the order of atomic sums: 1e-12 of the norm for one
application (a few hundred terms) and 1e-10 for a solve to 1e-8, as in the
graph tests; projections have no atomics, 1e-14.
"""
import numpy as np
import pytest

import pibem_amd as P
from pibem_amd import hip
from pibem_amd import mesh as M

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(b)


def take(f, pr):
    f.init_fma(pr.mesh, pr.dirichlet)
    f.generate_octree_blocking()
    f.direct_integrals()
    f.multipole_integrals()


def everything(f, pr):
    """What is called on one mesh, in an order that fills every kept buffer."""
    bp = P.BEMProblem(f)
    rng = np.random.default_rng(7)
    x = rng.uniform(-1, 1, (3, f.n))
    out = {"normals": bp.compute_normals()}
    bp.compute_alpha()
    dx, dy = hip.DeviceArray.from_numpy(x.ravel()), hip.DeviceArray(3 * f.n)
    for precision in (P.PBFMM_FP64, P.PBFMM_MIXED):
        for _ in range(60):  # past the application that times the plans
            bp.vmult_dev(dx.value, dy.value, precision)
    for plan in (4, 24, 92):  # slots, second stream
        f.set_side_fusion(P.PBFMM_FP64, plan)
        bp.vmult_dev(dx.value, dy.value, P.PBFMM_FP64)
        hip.synchronize()
        out[f"plan {plan}"] = dy.numpy()[:f.n]
    f.set_side_fusion(P.PBFMM_FP64, 4)
    bp.vmult_dev_multi(dx.value, dy.value, 3)
    hip.synchronize()
    out["vmult multi"] = dy.numpy()
    rhs = bp.compute_rhs(pr.tmp_rhs)
    db = hip.DeviceArray.from_numpy(np.concatenate([rhs, 0.5 * rhs, -rhs]))
    for graph in (0, 1):
        f.set_graph_mode(graph)
        sol = hip.DeviceArray(f.n)
        _, rr = f.gmres_dev(db.value, sol.value, 1e-8, 50, 500, P.PBFMM_FP64)
        assert rr <= 1e-8
        out[f"solve graph {graph}"] = sol.numpy()
    sol = hip.DeviceArray(f.n)
    _, rr = f.gmres_dev(db.value, sol.value, 1e-8, 50, 500, P.PBFMM_MIXED)
    assert rr <= 1e-8
    sol = hip.DeviceArray(3 * f.n)
    f.gmres_dev_multi(db.value, sol.value, 3, f.n, 1e-8, 50, 500, P.PBFMM_FP64)
    hip.synchronize()
    out["solve multi"] = sol.numpy()
    out["gradients"] = bp.compute_surface_gradients(pr.tmp_rhs)
    return out


def bar(name):
    return 1e-14 if name in ("normals", "gradients") else 1e-10 if name.startswith("solve") else 1e-12


@pytest.mark.parametrize("first,then", [((8, 1), (24, 1)), ((24, 1), (8, 1)), ((8, 1), (12, 2)), ((2, 1), (20, 1))])
def test_equals_a_new_handle(first, then):
    def problem(n, degree):
        return M.config_sphere(n, 4) if degree == 1 else M.config_spheroid(n, 4)

    a, b = problem(*first), problem(*then)
    assert (a.p, a.levels, a.max_nodes_per_leaf, a.sing_rule) == (b.p, b.levels, b.max_nodes_per_leaf, b.sing_rule)
    f = P.setup(a, P.PBFMM_MIXED)
    everything(f, a)
    print(f"\n[case] {a.mesh.name} N={a.mesh.n_dofs} then {b.mesh.name} N={b.mesh.n_dofs}", flush=True)
    f.set_graph_mode(-1)
    f.set_side_fusion(P.PBFMM_FP64, -1)
    f.set_side_fusion(P.PBFMM_MIXED, 24)
    take(f, b)
    st = f.tuning_state()
    assert st["side_fusion_fp64"] == -1 and st["side_fusion_fp32"] == 24  # the caller's plan stays
    assert st["graph_fp64"] == -1
    f.set_side_fusion(P.PBFMM_MIXED, -1)
    got = everything(f, b)
    new = P.setup(b, P.PBFMM_MIXED)
    want = everything(new, b)
    for k, w in want.items():
        print(f"  {k}: {rel(got[k], w):.1e}", flush=True)
        assert rel(got[k], w) <= bar(k), k
    f.close()
    new.close()


def test_refused_mesh_changes_nothing():
    """init_fma with a DoF out of range fails and leaves the handle with its mesh."""
    pr = M.config_sphere(8, 4)
    f = P.setup(pr, P.PBFMM_FP64)
    bp = P.BEMProblem(f)
    bp.compute_alpha()
    x = np.random.default_rng(3).uniform(-1, 1, f.n)
    y = bp.vmult(x)
    bad = M.config_sphere(12, 4)
    bad.mesh.cell_dofs = bad.mesh.cell_dofs.copy()
    bad.mesh.cell_dofs[0, 0] = bad.mesh.n_dofs
    with pytest.raises(P.PbfmmError):
        f.init_fma(bad.mesh, bad.dirichlet)
    assert rel(bp.vmult(x), y) <= 1e-12 and np.isfinite(bp.compute_normals()).all()
    f.close()
