"""Every truncation order against the oracle: each has its own expansion
length, tile count and split over wavefronts in the translations, with
partial chunks of pairs at every octree level.  Expansions, both kernels'
product and the operator in either precision, with M2L added to the targets
and in slots.  Bars as for the other parity tests: expansions 1e-11, FP64
products 1e-10, the FP32 operator 2e-5.
"""
import numpy as np
import pytest

import pibem_amd as P
from pibem_amd import mesh as M

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("order", range(1, 11))
def test_order_parity(oracle_mod, order):
    from pibem_amd import hip
    pr = M.config_sphere(10, order)
    print(f"\n[case] sphere N={pr.mesh.n_dofs} order={order}", flush=True)
    o, f = oracle_mod.OracleFMM(pr).setup(), P.setup(pr, P.PBFMM_MIXED)
    bp = P.BEMProblem(f)
    rng = np.random.default_rng(order)
    phi, dphi = rng.uniform(-1, 1, f.n), rng.uniform(-1, 1, f.n)
    o.generate_multipole_expansions(phi, dphi)
    N0, D0 = o.multipole_matr_vect_products(phi, dphi)
    f.generate_multipole_expansions(phi, dphi)
    me = f.expansions("me")
    N1, D1 = f.multipole_matr_vect_products(phi, dphi)
    for a, b in list(zip(o.expansions("me"), me)) + list(zip(o.expansions("le"), f.expansions("le"))):
        assert np.max(np.linalg.norm(a - b, axis=1)) <= 1e-11 * np.linalg.norm(a, axis=1).max()
    assert rel(N1, N0) <= 1e-10 and rel(D1, D0) <= 1e-10
    o.compute_alpha()
    bp.compute_alpha()
    v0 = o.vmult(phi)
    src, dst = hip.DeviceArray.from_numpy(phi), hip.DeviceArray(f.n)
    for precision, tol in ((P.PBFMM_FP64, 1e-10), (P.PBFMM_MIXED, 2e-5)):
        for plan in (0, 3, 4):
            f.set_side_fusion(precision, plan)
            bp.vmult_dev(src.value, dst.value, precision)
            hip.synchronize()
            e = rel(dst.numpy(), v0)
            print(f"  precision {precision} plan {plan}: {e:.1e}", flush=True)
            assert e <= tol
    f.close()
