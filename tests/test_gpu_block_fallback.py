"""Preconditioner blocks without an inverse become diagonal scaling.

One step of right-preconditioned GMRES from zero is x = a M^-1 b, a the
minimising factor, so the solution after one step shows M^-1 b up to a factor.
On the double-node cube without constraints the blocks that hold both copies
of a point have two equal rows; over their rows x must be a b / diag, over the
others' a times numpy's inverse of the exported block.

The FP64 inverses agree with numpy's to the blocks' condition numbers (below
1e4 for the invertible ones) times the rounding: 1e-10; mixed solves apply the
FP32 copies: 1e-5.
"""
import numpy as np
import pytest

import pibem_amd as P
from pibem_amd import hip
from pibem_amd import mesh as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,leaf", [(32, 20), (128, 20), (128, 1000)])
@pytest.mark.parametrize("precision,tol", [(P.PBFMM_FP64, 1e-10), (P.PBFMM_MIXED, 1e-5)])
def test_singular_blocks_scale_by_their_diagonal(rows, leaf, precision, tol):
    pr = M.config_dcube(6, 4)
    pr.max_nodes_per_leaf = leaf  # 1000: one block of 294 rows, above the largest that is inverted in LDS
    f = P.setup(pr, precision)
    f.set_preconditioner_rows(rows)
    bp = P.BEMProblem(f)
    bp.compute_alpha()
    blocks = bp.preconditioner_blocks()
    b = np.random.default_rng(1).uniform(-1, 1, f.n)
    want, singular = np.zeros(f.n), 0
    for idx, A in blocks:
        s = np.linalg.svd(A, compute_uv=False)
        if s[-1] <= 1e-12 * s[0]:
            singular += 1
            want[idx] = b[idx] / np.diag(A)
        else:
            assert s[-1] >= 1e-4 * s[0]
            want[idx] = np.linalg.solve(A, b[idx])
    db, dx = hip.DeviceArray.from_numpy(b), hip.DeviceArray.from_numpy(np.zeros(f.n))
    f.gmres_dev(db.value, dx.value, 1e-3, 1, 1, precision, check=False)
    x = dx.numpy()
    a = (x @ want) / (want @ want)
    e = np.linalg.norm(x - a * want) / np.linalg.norm(x)
    print(f"\n[case] cube N={f.n} {len(blocks)} blocks, {singular} without an inverse; off {e:.1e}", flush=True)
    assert singular > 0 and a != 0 and e <= tol
    f.close()
