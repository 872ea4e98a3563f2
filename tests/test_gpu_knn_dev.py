"""The device kNN on pitched arrays where a wave takes several queries: queries
in spatial order (which share a gathered list of points), in none (whose
results are written by the run) and half of each; remainders of a run."""
import numpy as np
import pytest
from test_gpu_knn import _Hip

pytestmark = pytest.mark.gpu


def knn_dev(vdn, ref, query, k, pitch_extra=0):
    nq = len(query)
    out = np.full((k, nq + pitch_extra), -7, dtype=np.int32)
    hip = _Hip()
    dev = [hip.to_dev(np.ascontiguousarray(x)) for x in (ref.T, query.T, out)]
    try:
        rc = vdn.lib().vd_knn_dev(dev[0], len(ref), len(ref), dev[1], nq, nq, 3, k, dev[2], nq + pitch_extra, None)
        assert rc == 0
        out = hip.to_host(dev[2], out)
    finally:
        for p in dev:
            hip.free(p)
    assert np.all(out[:, nq:] == -7)
    return out[:, :nq].T


def in_order(p):
    """p by cells of a coarse grid, boustrophedon within a layer."""
    c = (p / 40).astype(np.int64)
    y = np.where(c[:, 2] % 2 == 0, c[:, 1], 1000 - c[:, 1])
    x = np.where(y % 2 == 0, c[:, 0], 1000 - c[:, 0])
    return p[np.lexsort((x, y, c[:, 2]))]


@pytest.mark.parametrize("n_ref,n_query,k,order,refs", [
    (1500, 8192, 64, "random", "uniform"), (1500, 8193, 64, "spatial", "uniform"),
    (1500, 24575, 17, "mixed", "uniform"), (1500, 24577, 64, "mixed", "clusters"),
    (1200, 24583, 1, "random", "uniform"), (1200, 16385, 65, "random", "clusters"),
    (1200, 12289, 128, "spatial", "clusters"), (700, 8199, 130, "random", "uniform"),
    (300, 24581, 256, "mixed", "clusters"), (40, 24577, 64, "random", "uniform"),
])
def test_runs_of_pitched_queries(vdn, O, n_ref, n_query, k, order, refs):
    rng = np.random.default_rng(n_ref + 7 * n_query + k)
    ref = rng.random((n_ref, 3), dtype=np.float32) * 1000
    if refs == "clusters":
        at = rng.permutation(n_ref)[: n_ref // 2]
        ref[at] = 500 + 3 * rng.random((len(at), 3), dtype=np.float32)
        ref[at[:20]] = ref[at[0]]
    query = rng.random((n_query, 3), dtype=np.float32) * 1000
    query[rng.permutation(n_query)[: n_query // 8]] = ref[rng.integers(0, n_ref, n_query // 8)]
    if order == "spatial":
        query = in_order(query)
    elif order == "mixed":
        query[: n_query // 2] = in_order(query[: n_query // 2])
    got = knn_dev(vdn, ref, query, k, pitch_extra=5)
    want = O.knn(ref, query, k, False, grid=False)
    np.testing.assert_array_equal(got, want)
