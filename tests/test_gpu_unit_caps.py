"""The site-major clipping's work units at vertex caps and table depths that
leave pairs to the re-clip (the automatic ones of large problems, and smaller
ones, with more resident waves), every pair against the oracle bit for bit."""
import ctypes

import numpy as np
import pytest
from conftest import oracle_knn, problem
from test_gpu_knn import _Hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ns,tk,cfg", [
    (10, 600, 64, {"site_tcap": 17, "site_depth": 40}), (12, 1000, 64, {"site_tcap": 17, "site_depth": 40}),
    (10, 600, 64, {"site_tcap": 17, "site_depth": 8}), (10, 600, 64, {"site_tcap": 8, "site_depth": 8}),
    (10, 2, 2, {"site_tcap": 12, "site_depth": 40}), (14, 8200, 64, {"site_tcap": 17, "site_depth": 16}),
    (14, 8200, 64, {"site_tcap": 17, "site_depth": 40, "clip_blocks": 5000}),
    (10, 600, 20, {"site_tcap": 17, "site_depth": 40, "moments": "reference"}),
    (24, 8294, 64, {}),  # 386,000 pieces: the automatic caps, at first for unmoved sites
])
def test_units_at_small_caps(vdn, O, n, ns, tk, cfg):
    verts, tets, sites = problem("cube", n, ns)
    sk, tkn = oracle_knn("cube", n, ns, 90, tk)
    cfg = {"moments": "robust", **cfg}
    r = O.clip_tets(sites, sk, verts, tets, tkn, geom="f32", pair_acc="f64", site_mode=O.SITE_FIXED,
                    moments=cfg["moments"])
    with vdn.Engine(tet_k=tk, accum="f64", record_pairs=1, **cfg) as e:
        e.set_mesh(verts, tets)
        e.set_sites(sites)
        for _ in range(2):  # the second step at the depth of moved sites
            e.knn_step()
            e.clip_step()
            st, vals = e.pairs()
            np.testing.assert_array_equal(st.astype(np.int32), r["pair_status"])
            np.testing.assert_array_equal(vals, r["pair_vals"])
            np.testing.assert_array_equal(e.moments(), r["site_vals"])
            hist = e.status_hist()
            assert [hist[k] for k in vdn.STATUS_NAMES] == np.bincount(r["pair_status"], minlength=7).tolist()


@pytest.mark.parametrize("n,ns", [(10, 600), (24, 8294)])
def test_second_iteration_allocates_nothing(vdn, n, ns):
    """(An iteration that allocated could not be captured in a graph.)"""
    hip = _Hip()

    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.L.hipDeviceSynchronize() == 0
        assert hip.L.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    verts, tets, sites = problem("cube", n, ns)
    for moments in ("reference", "robust"):
        with vdn.Engine(tet_k=20, accum="f64", moments=moments) as e:
            e.set_mesh(verts, tets)
            e.set_sites(sites)
            e.lloyd(1)
            before = free()
            e.lloyd(2)
            assert free() == before
