"""The kNN grid's two builds (one workgroup for small instances, separate
passes for larger ones) and its in-cell order, light and crowded cells.

A grid lists its points by cell, then by input index, whatever builds it."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def points(n, crowd, seed):
    """n points of which `crowd` share a region much smaller than a cell; some coincide."""
    rng = np.random.default_rng(seed)
    p = rng.random((n, 3), dtype=np.float32) * 1000
    at = rng.permutation(n)[:crowd]
    p[at] = 437 + rng.random((crowd, 3), dtype=np.float32)
    p[at[: crowd // 8]] = p[at[0]] if crowd else 0
    return p


@pytest.mark.parametrize("n,crowd", [(2, 0), (65, 17), (1025, 1024), (8191, 3), (8192, 2500), (8193, 16), (8193, 17),
                                     (12000, 5000), (40000, 1025)])
def test_grid_order(vdn, O, n, crowd):
    p = points(n, crowd, 40 + n)
    k = min(8, n - 1)
    kn = vdn.KnProblem(p, k)
    kn.solve()
    perm = kn.permutation().astype(np.int64)
    np.testing.assert_array_equal(np.sort(perm), np.arange(n))
    np.testing.assert_array_equal(kn.points(), p[perm])
    i = kn.info()
    counts = np.zeros(i.dimx * i.dimy * i.dimz, dtype=np.int32)
    vdn.lib().vd_kn_get_cell_counts.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    assert vdn.lib().vd_kn_get_cell_counts(kn.h, counts.ctypes.data_as(ctypes.c_void_p)) == 0
    assert counts.sum() == n
    # inside every cell the ids ascend
    cell = np.repeat(np.arange(len(counts)), counts)
    assert np.all((np.diff(perm) > 0) | (np.diff(cell) > 0))
    if crowd:
        assert counts.max() >= crowd // 8
    np.testing.assert_array_equal(perm[kn.knearests().astype(np.int64)], O.knn(p, p, k, True, grid=False)[perm])
    kn.close()


@pytest.mark.parametrize("sizes", [(8192, 91), (8193, 200, 8192)])
def test_batch_grids(vdn, O, sizes):
    """Instances on both sides of the one-workgroup limit, each as alone."""
    from voronoi_amd import meshgen

    probs = [meshgen.make_problem("cube", 6, n, seed=60 + i) for i, n in enumerate(sizes)]
    with vdn.Engine(tet_k=16, site_k=20) as e:
        e.set_batch(probs)
        e.knn_step()
        sk, tk = e.site_knn(), e.tet_knn()
        off = e.batch_sites
    t0 = 0
    for i, (v, t, s) in enumerate(probs):
        np.testing.assert_array_equal(sk[off[i]:off[i + 1]] - off[i], O.site_knn(s, 20))
        np.testing.assert_array_equal(tk[t0:t0 + len(t)] - off[i], O.tet_knn(v, t, s, 16))
        t0 += len(t)


@pytest.mark.parametrize("n,k", [(4095, 90), (8191, 65), (8192, 20), (8193, 64), (12289, 90), (24577, 20)])
def test_runs_of_queries(vdn, O, n, k):
    """Query counts around the multiples of 4,096 at which a wave's run of
    queries grows from one to six; the second step starts from the first's rows."""
    from voronoi_amd import meshgen

    verts, tets, sites = meshgen.make_problem("cube", 5, n, seed=70 + n % 10)
    with vdn.Engine(tet_k=16, site_k=k, accum="f64") as e:
        e.set_mesh(verts, tets)
        e.set_sites(sites)
        for step in range(4):
            cur = e.sites()
            e.knn_step()
            print(f"{n} step {step}", flush=True)
            np.testing.assert_array_equal(e.site_knn(), O.site_knn(cur, k))
            np.testing.assert_array_equal(e.tet_knn(), O.tet_knn(verts, tets, cur, 16))
            e.clip_step()
            e.update_step()
