"""Kernel B with a wavefront per site: cells of few and many vertices, launch
caps that cells reach, one site, duplicate sites, every pair of the cell form
against the oracle bit for bit."""
import numpy as np
import pytest
from conftest import problem

pytestmark = pytest.mark.gpu


def check(vdn, O, verts, tets, sites, tk, **cfg):
    k = min(90, len(sites) - 1)
    tk = min(tk, len(sites))
    sk, tkn = O.site_knn(sites, k), O.tet_knn(verts, tets, sites, tk)
    caps = {n: cfg[n] for n in ("pcap", "tcap") if n in cfg}
    r = O.clip_cells(sites, sk, verts, tets, tkn, geom="f32", pair_acc="f64", site_mode=O.SITE_FIXED, moments="robust",
                     **caps)
    with vdn.Engine(form="cells", tet_k=tk, accum="f64", moments="robust", record_pairs=1, **cfg) as e:
        e.set_mesh(verts, tets)
        e.set_sites(sites)
        e.knn_step()
        e.clip_step()
        st, vals = e.pairs()
        np.testing.assert_array_equal(st.astype(np.int32), r["pair_status"])
        np.testing.assert_array_equal(vals, r["pair_vals"])
        np.testing.assert_array_equal(e.moments(), r["site_vals"])


@pytest.mark.parametrize("n,ns,tk,cfg", [
    (4, 2, 2, {}), (4, 5, 5, {}), (6, 66, 20, {}), (9, 255, 40, {}), (10, 257, 40, {}),
    (9, 300, 40, {"cells_pcap": 20, "cells_tcap": 30}), (9, 300, 40, {"cells_pcap": 64, "cells_tcap": 96}),
    (9, 300, 40, {"pcap": 80, "tcap": 120}), (9, 300, 40, {"pcap": 30, "tcap": 40}),
])
def test_cells_bit_exact(vdn, O, n, ns, tk, cfg):
    verts, tets, sites = problem("cube", n, ns)
    check(vdn, O, verts, tets, sites, tk, **cfg)


def test_cells_of_many_planes(vdn, O):
    """Sites on two concentric shells: the inner cells have more than 64 vertices."""
    rng = np.random.default_rng(8)
    u = rng.standard_normal((160, 3))
    u /= np.linalg.norm(u, axis=1)[:, None]
    sites = np.concatenate([[[500, 500, 500]], 500 + 300 * u * (1 + 0.01 * rng.random((160, 1)))]).astype(np.float32)
    verts, tets, _ = problem("cube", 5, 10)
    check(vdn, O, verts, tets, sites, 30)
    check(vdn, O, verts, tets, sites, 30, pcap=70, tcap=130)


def test_cells_of_duplicate_sites(vdn, O):
    verts, tets, sites = problem("cube", 5, 60)
    sites = np.concatenate([sites, sites[:7]])
    check(vdn, O, verts, tets, sites, 30)
