"""The site-major clipping's work units: sites with fewer and more pairs than a
unit holds, on both sides of the unit size's change, every pair against the
oracle bit for bit."""
import numpy as np
import pytest
from conftest import oracle_knn, problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ns,tk,cull", [(10, 2, 64, 16), (10, 2, 64, 0), (11, 60, 60, 0), (9, 700, 64, 16),
                                          (14, 8191, 64, 16), (14, 8192, 64, 0)])
def test_units_bit_exact(vdn, O, n, ns, tk, cull):
    verts, tets, sites = problem("cube", n, ns)
    sk, tkn = oracle_knn("cube", n, ns, 90, tk)
    r = O.clip_tets(sites, sk, verts, tets, tkn, geom="f32", pair_acc="f64", site_mode=O.SITE_FIXED, moments="robust")
    with vdn.Engine(tet_k=tk, accum="f64", moments="robust", record_pairs=1, cull_depth=cull) as e:
        e.set_mesh(verts, tets)
        e.set_sites(sites)
        for _ in range(2):  # the second step at the moved sites' table depth
            e.knn_step()
            e.clip_step()
            st, vals = e.pairs()
            mom, hist = e.moments(), e.status_hist()
            np.testing.assert_array_equal(st.astype(np.int32), r["pair_status"])
            np.testing.assert_array_equal(vals, r["pair_vals"])
            np.testing.assert_array_equal(mom, r["site_vals"])
            assert [hist[k] for k in vdn.STATUS_NAMES] == np.bincount(r["pair_status"], minlength=7).tolist()
