"""Near-field assembly against the oracle where its tiles change: leaves of
fewer rows than a tile, a remainder of rows, more columns than one tile, quad
rules of 1 to 64 points (the entry masks' width), mirrored cells, both
singular rules, nodes with several doubles, and more singular items in a tile
than its list holds.

Entries are single sums of at most 64 terms per cell of at most a few cells,
evaluated with reciprocal square roots and fused multiply-adds here and
separately rounded operations there: 1e-12 of the largest entry, as the
near field's own test.
"""
import numpy as np
import pytest

import pibem_amd as P
from pibem_amd import mesh as M

pytestmark = pytest.mark.gpu


def problem(m, **kw):
    d = np.zeros(m.n_dofs, np.uint8)
    d[m.cell_dofs[M.cell_centroids(m)[:, 2] > 0].ravel()] = 1
    return M.Problem(m, d, None, np.zeros(m.n_dofs), 2, **kw)


def fan(sheets=7, cells=10, extra=3):
    """Kite-shaped quads around one point, the point and the ring edges doubled between sheets: the `sheets`
    doubles of the point each see every cell."""
    n = sheets * cells
    ang = 2 * np.pi * np.arange(2 * n + 1) / (2 * n)
    cone = lambda r, a: np.array([r * np.cos(a), r * np.sin(a), 0.3 * r * r])  # noqa: E731
    pts, quads = [], []
    for s in range(sheets):
        pole = len(pts)
        pts.append(cone(0.0, 0.0))
        for k in range(cells + 1):
            pts.append(cone(1.0, ang[2 * (s * cells + k)]))
        for k in range(cells):
            pts.append(cone(1.6, ang[2 * (s * cells + k) + 1]))
        for k in range(cells):
            quads.append([pole, pole + 1 + k, pole + 2 + k, pole + 2 + cells + k])
    xyz = np.array(pts)
    m = M.Mesh(xyz, np.array(quads, dtype=np.int64), 4, np.tile([0.0, 0.0, 1.0], (len(pts), 1)),
               np.zeros(len(quads), np.int32), name="fan")
    m.dbl_ptr, m.dbl_idx = M._double_nodes(xyz)
    return m


CASES = [
    ("few rows per leaf", lambda: problem(M.cube_sphere(12, 1), max_nodes_per_leaf=4)),
    ("wide leaves", lambda: problem(M.cube_sphere(16, 1), max_nodes_per_leaf=500)),
    ("wide Q2 leaves", lambda: problem(M.cube_sphere(7, 2, (2.0, 1.0, 1.0)), max_nodes_per_leaf=150)),
    ("one point", lambda: problem(M.cube_sphere(6, 1), quad_order=1)),
    ("36 points", lambda: problem(M.cube_sphere(5, 2), quad_order=6)),
    ("64 points, Telles", lambda: problem(M.cube_sphere(6, 1), quad_order=8, sing_rule=0)),
    ("double nodes", lambda: problem(M.double_node_cube(6))),
    ("mirrored hull", lambda: problem(M.wigley_hull(30, 4, z_top=0.0), mirror_z0=0.0)),
    ("many singular cells at a point", lambda: problem(fan(), max_nodes_per_leaf=200)),
]


@pytest.mark.parametrize("name,make", CASES, ids=[c[0] for c in CASES])
def test_nearfield(oracle_mod, name, make):
    pr = make()
    print(f"\n[case] {name} N={pr.mesh.n_dofs} cells={pr.mesh.n_cells}", flush=True)
    o = oracle_mod.OracleFMM(pr).setup()
    f = P.setup(pr, P.PBFMM_FP64)
    rp, col, vN, vD, _ = o.csr()
    grp, gcol, gN, gD = f.nearfield(P.PBFMM_FP64)
    f.close()
    assert np.array_equal(rp, grp) and np.array_equal(col, gcol)
    eN, eD = np.max(np.abs(gN - vN)) / np.max(np.abs(vN)), np.max(np.abs(gD - vD)) / np.max(np.abs(vD))
    print(f"  N {eN:.1e} D {eD:.1e}", flush=True)
    assert eN <= 1e-12 and eD <= 1e-12
