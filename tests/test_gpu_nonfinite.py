"""A site whose coordinates are infinite, NaN or so large that its bisectors'
FP32 coefficients overflow, among a seed's first neighbours: the emptiness test
may not drop a pair for such a bisector."""
import numpy as np
import pytest
from conftest import problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["site", "cells"])
@pytest.mark.parametrize("n_sites", [2, 5, 17])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan, 1e36, 3e35, 1e18])
def test_emptiness_pass_with_a_site_out_of_range(vdn, O, bad, n_sites, form):
    """Every pair with the test equals the pair without it, and the oracle's
    where the sites' order by distance is the oracle's too (not with NaN) and
    the site's own bisectors are (not at -inf)."""
    verts, tets, sites = problem("cube", 4, n_sites)
    b = n_sites // 2
    sites = sites.copy()
    sites[b, 0] = bad

    def run(depth):
        with vdn.Engine(form=form, tet_k=n_sites, accum="f64", moments="robust", record_pairs=1,
                        cull_depth=depth) as e:
            e.set_mesh(verts, tets)
            e.set_sites(sites)
            e.knn_step()
            e.clip_step()
            return (*e.pairs(), e.moments(), e.site_knn(), e.tet_knn())

    st, vals, mom, sk, tk = run(16)
    for got, want in zip((st, vals, mom), run(0)):
        np.testing.assert_array_equal(got, want)
    if not bad > 0:
        return
    clip = O.clip_cells if form == "cells" else O.clip_tets
    r = clip(sites, sk, verts, tets, tk, geom="f32", pair_acc="f64", site_mode=O.SITE_FIXED, moments="robust")
    np.testing.assert_array_equal(st.astype(np.int32), r["pair_status"])
    fin = tk.ravel() != b  # (the site's own pieces have no meaningful sums)
    np.testing.assert_array_equal(vals[fin], r["pair_vals"][fin])
    np.testing.assert_array_equal(np.delete(mom, b, 0), np.delete(r["site_vals"], b, 0))


@pytest.mark.parametrize("form", ["site", "cells"])
def test_emptiness_pass_beside_an_unused_nan_vertex(vdn, O, form):
    """Tets of a frame of a million units whose tips lie within the FP32
    rounding of a bisector through the origin, with a vertex that no tet uses
    at NaN: the test's rounding bound comes from the tets' own corners."""
    rng = np.random.default_rng(3)
    a = np.array([300000.0, 410000.0, -230000.0], np.float32)
    sites = np.stack([a, -a])
    u = a.astype(np.float64) / np.linalg.norm(a.astype(np.float64))
    w = np.cross(u, [0, 0, 1.0])
    w /= np.linalg.norm(w)
    x = np.cross(u, w)
    m = 4000
    p = rng.uniform(-1e6, 1e6, (m, 3))
    p -= np.outer(p @ u, u)
    corners = [p + rng.uniform(0, 0.1, (m, 1)) * u]
    corners += [p - 8 * u + 4 * (np.cos(t) * w + np.sin(t) * x) for t in (0.0, 2.1, 4.2)]
    verts = np.stack(corners, 1).astype(np.float32).reshape(-1, 3)
    verts = np.concatenate([np.full((1, 3), np.nan, np.float32), verts])
    tets = 1 + np.arange(4 * m, dtype=np.int32).reshape(m, 4)

    def run(depth):
        with vdn.Engine(form=form, tet_k=2, accum="f64", moments="robust", record_pairs=1, cull_depth=depth) as e:
            e.set_mesh(verts, tets)
            e.set_sites(sites)
            e.knn_step()
            e.clip_step()
            return (*e.pairs(), e.site_knn(), e.tet_knn())

    st, vals, sk, tk = run(16)
    for got, want in zip((st, vals), run(0)):
        np.testing.assert_array_equal(got, want)
    clip = O.clip_cells if form == "cells" else O.clip_tets
    r = clip(sites, sk, verts, tets, tk, geom="f32", pair_acc="f64", site_mode=O.SITE_FIXED, moments="robust")
    np.testing.assert_array_equal(st.astype(np.int32), r["pair_status"])
