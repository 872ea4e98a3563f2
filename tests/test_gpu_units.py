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


@pytest.mark.parametrize("n,ns", [(3, 40), (21, 5000), (21, 5800)])
def test_small_problem_caps(vdn, O, n, ns):
    """The automatic caps below and above the small-problem limit (256,000
    estimated pieces: 55,566 tets with 5,000 and 5,800 sites lie on its two
    sides) and the same caps given by hand: one result, the oracle's."""
    verts, tets, sites = problem("cube", n, ns)
    tk = min(64, ns)
    sk, tkn = oracle_knn("cube", n, ns, 90, tk)
    r = O.clip_tets(sites, sk, verts, tets, tkn, geom="f32", pair_acc="f64", site_mode=O.SITE_FIXED, moments="robust",
                    want_pairs=False)
    for cfg in ({}, {"site_tcap": 32, "site_depth": 90}, {"site_tcap": 17, "site_depth": 40}):
        with vdn.Engine(tet_k=tk, accum="f64", moments="robust", **cfg) as e:
            e.set_mesh(verts, tets)
            e.set_sites(sites)
            e.knn_step()
            e.clip_step()
            np.testing.assert_array_equal(e.moments(), r["site_vals"])


@pytest.mark.parametrize("n,ns,tk", [(22, 6389, 20), (12, 9000, 20), (8, 3000, 64)])
def test_records_at_few_candidates(vdn, O, n, ns, tk):
    """More pieces than a tenth of the pairs (few candidates, dense sites)."""
    verts, tets, sites = problem("cube", n, ns)
    sk, tkn = oracle_knn("cube", n, ns, 90, tk)
    for moments in ("reference", "robust"):
        r = O.clip_tets(sites, sk, verts, tets, tkn, geom="f32", pair_acc="f64", site_mode=O.SITE_FIXED,
                        moments=moments, want_pairs=False)
        with vdn.Engine(tet_k=tk, accum="f64", moments=moments) as e:
            e.set_mesh(verts, tets)
            e.set_sites(sites)
            e.knn_step()
            e.clip_step()
            np.testing.assert_array_equal(e.moments(), r["site_vals"])


@pytest.mark.parametrize("n,ns,tk,depth", [(5, 30, 30, 1), (9, 2048, 40, 16), (9, 2049, 40, 16), (8, 90, 64, 2),
                                           (12, 400, 33, 90)])
def test_emptiness_pass_bit_exact(vdn, O, n, ns, tk, depth):
    """The emptiness pass with one and four waves per site, at few and many
    bisectors, at candidate counts that are and are not powers of two."""
    verts, tets, sites = problem("cube", n, ns)
    sk, tkn = oracle_knn("cube", n, ns, 90, tk)
    r = O.clip_tets(sites, sk, verts, tets, tkn, geom="f32", pair_acc="f64", site_mode=O.SITE_FIXED, moments="robust")
    with vdn.Engine(tet_k=tk, accum="f64", moments="robust", record_pairs=1, cull_depth=depth) as e:
        e.set_mesh(verts, tets)
        e.set_sites(sites)
        e.knn_step()
        e.clip_step()
        st, vals = e.pairs()
        np.testing.assert_array_equal(st.astype(np.int32), r["pair_status"])
        np.testing.assert_array_equal(vals, r["pair_vals"])
        np.testing.assert_array_equal(e.moments(), r["site_vals"])
        hist = e.status_hist()
        assert [hist[k] for k in vdn.STATUS_NAMES] == np.bincount(r["pair_status"], minlength=7).tolist()
