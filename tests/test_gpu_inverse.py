"""The block-Jacobi inverses, through the solves they precondition: odd block
sizes (the padding of the stored column vectors), blocks close to the largest
one inverted in LDS (128 rows) and leaves above it, constrained rows, and
blocks without an inverse.

Where one block holds every row, the near field is the whole operator and its
inverse solves the system at once.  Otherwise right-preconditioned GMRES in
numpy, on the operator's own matrix (the GPU operator applied to the unit
vectors) with numpy's inverses of the exported blocks, takes the number of
steps that an exact inverse takes; the GPU's count may exceed it by the steps
it enqueues ahead of its stopping test (at most 2 here).
"""
import numpy as np
import pytest

import pibem_amd as P
from pibem_amd import hip
from pibem_amd import mesh as M

pytestmark = pytest.mark.gpu


def gmres_steps(A, Minv, b, tol):
    """Steps of right-preconditioned GMRES from zero until the residual is tol |b|."""
    n, beta = len(b), np.linalg.norm(b)
    V, H = [b / beta], np.zeros((61, 60))
    for k in range(60):
        w = A @ (Minv @ V[k])
        for _ in range(2):
            for i, v in enumerate(V):
                d = v @ w
                H[i, k] += d
                w -= d * v
        H[k + 1, k] = np.linalg.norm(w)
        e = np.zeros(k + 2)
        e[0] = beta
        y = np.linalg.lstsq(H[:k + 2, :k + 1], e, rcond=None)[0]
        if np.linalg.norm(e - H[:k + 2, :k + 1] @ y) <= tol * beta:
            return k + 1
        V.append(w / H[k + 1, k])
    return 60


@pytest.mark.parametrize("n,leaf,largest", [(2, 1000, 26), (3, 1000, 56), (4, 1000, 98), (12, 2000, 127),
                                            (16, 1000, 1000), (9, 20, 128)])
@pytest.mark.parametrize("precision", [P.PBFMM_FP64, P.PBFMM_MIXED])
def test_steps_of_an_exact_inverse(n, leaf, largest, precision):
    pr = M.config_sphere(n, 4)
    pr.max_nodes_per_leaf = leaf
    f = P.setup(pr, precision)
    bp = P.BEMProblem(f)
    bp.compute_alpha()
    N = f.n
    rhs = bp.compute_rhs(pr.tmp_rhs)
    blocks = bp.preconditioner_blocks()
    sizes = [len(r) for r, _ in blocks]
    x, y = hip.DeviceArray.from_numpy(np.eye(N).ravel()), hip.DeviceArray(N * N)
    bp.vmult_dev_multi(x.value, y.value, N)
    hip.synchronize()
    A = y.numpy().reshape(N, N).T
    Minv = np.zeros((N, N))
    for rows, B in blocks:
        Minv[np.ix_(rows, rows)] = np.linalg.inv(B)
    want = gmres_steps(A, Minv, rhs, 0.5e-8)
    db, dx = hip.DeviceArray.from_numpy(rhs), hip.DeviceArray(N)
    it, rr = f.gmres_dev(db.value, dx.value, 1e-8, 60, 200, precision)
    f.close()
    print(f"\n[case] N={N} blocks {min(sizes)}..{max(sizes)} steps {it}, numpy {want}, relres {rr:.1e}", flush=True)
    assert max(sizes) <= largest and (leaf < 1000 or len(sizes) == 1 or max(sizes) > 90)
    assert rr <= 1e-8
    # mixed: refinement repeats a few steps per inner solve
    assert it <= want + (2 if precision == P.PBFMM_FP64 else 4)


def test_constrained_rows():
    pr = M.config_dcube(5, 4)
    cons = M.constraints(pr)
    pr.max_nodes_per_leaf = 1000
    f = P.setup(pr)
    bp = P.BEMProblem(f)
    bp.compute_alpha()
    bp.set_constraints(cons)
    blocks = bp.preconditioner_blocks()
    ptr, idx, val, inh, isc = cons
    for rows, A in blocks:
        where = {int(d): k for k, d in enumerate(rows)}
        for k, d in enumerate(rows):
            if isc[d]:
                want = np.zeros(len(rows))
                want[k] = 1.0
                for q in range(ptr[d], ptr[d + 1]):
                    if int(idx[q]) in where:
                        want[where[int(idx[q])]] -= val[q]
                assert np.array_equal(A[k], want)
    _, _, it, rr = bp.solve_system(pr.tmp_rhs, 1e-8)
    f.close()
    print(f"\n[case] double-node cube N={pr.mesh.n_dofs} steps {it} relres {rr:.1e}", flush=True)
    assert rr <= 1e-8


def test_block_without_inverse():
    """Unconstrained doubles have equal rows, so the blocks that hold them have no inverse: diagonal scaling."""
    pr = M.config_dcube(3, 4)
    f = P.setup(pr, P.PBFMM_FP64)
    bp = P.BEMProblem(f)
    blocks = bp.preconditioner_blocks()
    assert min(np.linalg.matrix_rank(A) - len(A) for _, A in blocks) < 0
    b, y = hip.DeviceArray.from_numpy(np.random.default_rng(1).uniform(-1, 1, f.n)), hip.DeviceArray(f.n)
    it, rr = f.gmres_dev(b.value, y.value, 1e-3, 20, 20, check=False)
    print(f"\n[case] unconstrained cube: steps {it} relres {rr:.1e}", flush=True)
    assert np.isfinite(y.numpy()).all() and np.isfinite(rr)
    f.close()
