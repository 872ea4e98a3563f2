"""A device with memory for an iteration but not for the automatic record
buffer of all estimated pieces, or for the emptiness pass's second list: the
iteration runs with fewer records, or with one list."""
import ctypes

import numpy as np
import pytest
from conftest import problem
from test_gpu_knn import _Hip

pytestmark = pytest.mark.gpu

MB = 1 << 20


def _free(hip):
    a, b = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.L.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
    return a.value


def _fill(hip, leave):
    """Device buffers that leave about `leave` bytes free."""
    held = []
    size = 64 << 30
    while size >= 16 * MB:
        p = ctypes.c_void_p()
        if _free(hip) < leave + size:
            size //= 2
        elif hip.L.hipMalloc(ctypes.byref(p), size) == 0:
            held.append(p)
        else:  # (free, but not in one piece)
            hip.L.hipGetLastError()
            size //= 2
    return held


@pytest.mark.parametrize("n_sites,tet_k,least,short", [(129600, 8, 900, 300), (2000, 96, 3000, 250)])
def test_fewer_buffers_where_memory_is_short(vdn, n_sites, tet_k, least, short):
    verts, tets, sites = problem("cube", 60, n_sites)
    cfg = dict(tet_k=tet_k, accum="f64", moments="reference")

    small = problem("cube", 10, 600)
    hip = _Hip()

    def run(short_of):
        """The results and the device bytes of a context that has run before,
        with that many bytes too few."""
        with vdn.Engine(**cfg) as e:
            e.set_mesh(*small[:2])
            e.set_sites(small[2])
            e.lloyd(2)
            e.sync()
            free = _free(hip)
            held = _fill(hip, used - short_of) if short_of else []
            try:
                e.set_mesh(verts, tets)
                e.set_sites(sites)
                e.lloyd(2)
                return (e.moments(), e.sites()), free - _free(hip)
            finally:
                for p in held:
                    hip.free(p)

    want, used = run(0)
    # at 129,600 sites the records of the estimated pieces take 650 MB more than
    # those of one pair in ten; at 2,000 the second list takes 497 MB
    assert used > least * MB
    got, _ = run(short * MB)
    for a, b in zip(got, want):
        np.testing.assert_array_equal(a, b)
