"""generate + products on host vectors, whose SpMV runs on the second stream
from 1 M values on, with M2L on one workgroup per CU where values are many
for the M2L pairs, against the device call, which runs them in order.

The two add the same terms in another order: a few hundred per row, 1e-13 of
the vector's norm.
"""
import numpy as np
import pytest

import pibem_amd as P
from pibem_amd import mesh as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,order,leaf", [(16, 4, 20), (32, 6, 64), (40, 5, 400), (64, 4, 250), (64, 8, 20)])
def test_products_equal_device_call(n, order, leaf):
    from pibem_amd import hip
    pr = M.config_sphere(n, order)
    pr.max_nodes_per_leaf = leaf
    f = P.setup(pr)
    w = f.work_counts()
    print(f"\n[case] sphere N={f.n} order={order} leaf={leaf} values per pair "
          f"{w['near_values'] / max(w['m2l_pairs'], 1):.0f} {w}", flush=True)
    rng = np.random.default_rng(n)
    phi, dphi = rng.uniform(-1, 1, f.n), rng.uniform(-1, 1, f.n)
    d = [hip.DeviceArray.from_numpy(phi), hip.DeviceArray.from_numpy(dphi), hip.DeviceArray(f.n), hip.DeviceArray(f.n)]
    f.matvec_dev(d[0].value, d[1].value, d[2].value, d[3].value)
    hip.synchronize()
    for _ in range(3):  # one stream's work must not overtake the other's
        f.generate_multipole_expansions(phi, dphi)
        for got, want in zip(f.multipole_matr_vect_products(phi, dphi), d[2:]):
            want = want.numpy()
            e = np.linalg.norm(got - want) / np.linalg.norm(want)
            print(f"  {e:.1e}", flush=True)
            assert e <= 1e-13
    f.close()
