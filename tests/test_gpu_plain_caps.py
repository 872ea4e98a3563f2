"""The tet-major clip at caps where it keeps the vertices' distances and where it
does not (they would cost a resident wave, or do not fit the LDS): every pair
against the oracle bit for bit, with and without the arithmetic filter."""
import numpy as np
import pytest
from conftest import oracle_knn, problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pcap,tcap", [(64, 96), (32, 64), (40, 64), (100, 140), (12, 18)])
@pytest.mark.parametrize("filt", [0, 2])
def test_plain_caps_bit_exact(vdn, O, pcap, tcap, filt):
    verts, tets, sites = problem("cube", 8, 300)
    sk, tkn = oracle_knn("cube", 8, 300, 90, 64)
    r = O.clip_tets(sites, sk, verts, tets, tkn, geom="f32", pair_acc="f64", site_mode=O.SITE_FIXED, moments="robust",
                    pcap=pcap, tcap=tcap, filter=filt)
    with vdn.Engine(tet_k=64, form="tet", accum="f64", moments="robust", record_pairs=1, pcap=pcap, tcap=tcap,
                    filter=filt) as e:
        e.set_mesh(verts, tets)
        e.set_sites(sites)
        e.knn_step()
        e.clip_step()
        st, vals = e.pairs()
        np.testing.assert_array_equal(st.astype(np.int32), r["pair_status"])
        np.testing.assert_array_equal(vals, r["pair_vals"])
        np.testing.assert_array_equal(e.moments(), r["site_vals"])
