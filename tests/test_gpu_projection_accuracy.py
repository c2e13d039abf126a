"""How far the mass-matrix CG of the L2 projections goes past its tolerance.

The residual is tested after every eighth step, so a solve takes the first
multiple of eight steps whose residual is below 1e-13.  The same rule in numpy
on the oracle's mass matrix gives the steps to expect and the error E that is
left against a direct solve.  The GPU's error may be 4 E (another order of the
same sums) + 2e-14, the rounding of the direct solve (condition numbers up to
1e2): a solve that ends at its first residual below 1e-13 is up to 3e-13 off
on these meshes.  The cell normals are projected, whose integrals have no
cancellation on stretched cells; a surface gradient's metric loses six digits
there, on either side.
"""
import numpy as np
import pytest

import pibem_amd as P
from pibem_amd import mesh as M

pytestmark = pytest.mark.gpu


def cg_by_eights(A, b):
    """Jacobi CG on the columns of b until, after a multiple of eight steps, every |r| <= 1e-13 |b|."""
    d = A.diagonal()[:, None]
    x, r = np.zeros_like(b), b.copy()
    z = r / d
    p, rz, k = z.copy(), (r * z).sum(0), 0
    bb = (b * b).sum(0)
    while k == 0 or k % 8 or not ((r * r).sum(0) <= 1e-26 * bb).all():
        q = A @ p
        a = rz / np.where((p * q).sum(0) > 0, (p * q).sum(0), 1.0)
        x, r = x + a * p, r - a * q
        z = r / d
        new = (r * z).sum(0)
        p, rz = z + new / np.where(rz > 0, rz, 1.0) * p, new
        k += 1
    return x, k


@pytest.mark.parametrize("n,deg,radii", [(8, 2, (4.0, 1.0, 1.0)), (16, 2, (4.0, 1.0, 1.0)), (32, 1, (4.0, 1.0, 1.0)),
                                         (20, 1, (100.0, 1.0, 0.1)), (10, 2, (100.0, 1.0, 0.1))])
def test_steps_and_error(n, deg, radii):
    from orc_postsolve import PostSolve
    m = M.cube_sphere(n, deg, radii)
    f = P.BEMFMA(trunc_order=2)
    f.init_fma(m, np.ones(m.n_dofs, np.uint8))
    bp = P.BEMProblem(f)
    o = PostSolve(m)
    want = o.compute_normals()
    loc = np.einsum("iq,cqd,cq->cdi", o.N, o.n, o.JxW)
    b = np.zeros((m.n_dofs, 3))
    for d in range(3):
        np.add.at(b[:, d], m.cell_dofs.ravel(), loc[:, d, :].ravel())
    x, steps = cg_by_eights(o.M.tocsr(), b)
    err = np.linalg.norm(x.T.ravel() - want) / np.linalg.norm(want)
    got = np.linalg.norm(bp.compute_normals() - want) / np.linalg.norm(want)
    print(f"\n[case] q{deg} N={m.n_dofs} radii {radii}: steps {bp.projection_iterations()}, numpy {steps}; "
          f"error {got:.1e}, numpy {err:.1e}", flush=True)
    assert bp.projection_iterations() == steps
    assert got <= 4 * err + 2e-14
    f.close()
