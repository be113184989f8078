"""Fattening and link storage at the edges of their launches (slabs that are no
multiple of a block, several tiles, the smallest lattice) for every coefficient
pattern that takes its own kernels, against the oracle: relative L2 <= 1e-13,
the rounding of some twenty products of nearly unitary matrices."""
import numpy as np
import pytest

import qopqdp_amd as q
from conftest import MILC, gauge_numpy

pytestmark = pytest.mark.gpu
ZERO = dict(one_link=0.0, three_staple=0.0, five_staple=0.0, seven_staple=0.0, lepage=0.0, naik=0.0)
SETS = {
    "milc": MILC,
    "one_link": dict(ZERO, one_link=0.7),
    "three": dict(ZERO, one_link=0.1, three_staple=0.3),
    "five": dict(ZERO, five_staple=0.2, naik=0.1),
    "seven": dict(ZERO, three_staple=0.1, seven_staple=0.2),
    "lepage": dict(ZERO, lepage=0.25),
    "five_lepage": dict(ZERO, one_link=0.5, five_staple=0.1, lepage=-0.05, naik=-0.04),
    "fat7": dict(MILC, lepage=0.0, naik=0.0),
}


@pytest.mark.parametrize("L", [[4, 4, 4, 4], [4, 6, 10, 6], [6, 4, 4, 14]])
@pytest.mark.parametrize("name", list(SETS))
def test_fattened_links_match_oracle(oracle, L, name):
    U = gauge_numpy(L, 77, 0.4)
    oracle.rephase_milc(L, U)
    fat, lng = oracle.make_imp_links(L, U, SETS[name])
    s = q.Session(L)
    try:
        g = s.gauge(U)
        fla, info = s.links_from_gauge(g, SETS[name])
        assert info.status == 0
        naik = SETS[name]["naik"] != 0
        gf, gl = s.extract_links(fla, naik)
        for mu in range(4):
            assert np.linalg.norm(gf[mu] - fat[mu]) <= 1e-13 * np.linalg.norm(fat[mu])
            if naik:
                assert np.linalg.norm(gl[mu] - lng[mu]) <= 1e-13 * np.linalg.norm(lng[mu])
        v = q.gen_source(L, 78, q.QOP_EVENODD)  # the backward links too
        out, src = s.zeros(), s.vec(v)
        s.lib.QOP_D3_asqtad_dslash(None, fla, 0.1, out, src, 2, 2)
        h = oracle.links(L, fat, lng if naik else None)
        want = oracle.dslash(h, 0.1, v, 2, 2)
        assert np.linalg.norm(s.get(out) - want) <= 2e-13 * np.linalg.norm(want)
        oracle.free_links(h)
        s.free(out)
        s.free(src)
        s.lib.QOP_D3_asqtad_destroy_L(fla)
        s.lib.QOP_D3_destroy_G(g)
    finally:
        s.close()


def test_several_tiles(oracle):
    L = [4, 10, 14, 32]  # a slab of 2240 positions: two tiles of 1152
    U = gauge_numpy(L, 79, 0.4)
    fat, lng = oracle.make_imp_links(L, U, MILC)
    s = q.Session(L)
    try:
        g = s.gauge(U)
        fla, _ = s.links_from_gauge(g)
        gf, gl = s.extract_links(fla)
        for mu in range(4):
            assert np.linalg.norm(gf[mu] - fat[mu]) <= 1e-13 * np.linalg.norm(fat[mu])
            assert np.linalg.norm(gl[mu] - lng[mu]) <= 1e-13 * np.linalg.norm(lng[mu])
        s.lib.QOP_D3_asqtad_destroy_L(fla)
        s.lib.QOP_D3_destroy_G(g)
    finally:
        s.close()
