"""The mass-matrix CG of the L2 projections where its launches change shape:
fewer rows than one workgroup takes, a remainder of rows, more rows than one
pass of all workgroups (more than 32,768), both elements; zero data, and
components that converge in different steps.

Both sides solve the same mass matrix, the GPU to a relative residual of 1e-13
per component, the oracle directly; the mass matrix's condition number stays
below 1e3 on these meshes, so the two agree to 1e-10.
"""
import numpy as np
import pytest

import pibem_amd as P
from pibem_amd import mesh as M

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("n,deg", [(2, 1), (3, 2), (8, 1), (23, 1), (80, 1), (42, 2)])
def test_projection(n, deg):
    from orc_postsolve import PostSolve
    m = M.cube_sphere(n, deg, (2.0, 1.0, 1.0))
    N = m.n_dofs
    print(f"\n[case] projection n={n} q{deg} N={N}", flush=True)
    f = P.BEMFMA(trunc_order=2)
    f.init_fma(m, np.ones(N, np.uint8))
    bp = P.BEMProblem(f)
    o = PostSolve(m)
    assert rel(bp.compute_normals(), o.compute_normals()) <= 1e-10
    steps = bp.projection_iterations()
    assert 0 < steps < 200
    x = m.support_xyz
    phi = x[:, 0] ** 2 + np.sin(3.0 * x[:, 2])
    assert rel(bp.compute_surface_gradients(phi), o.compute_surface_gradients(phi)) <= 1e-10
    assert not bp.compute_surface_gradients(np.zeros(N)).any()
    assert bp.projection_iterations() == 0
    f.close()
