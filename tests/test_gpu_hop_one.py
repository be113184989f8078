"""The one-RHS hop of the reference path at the edges of its launches: the
four-wave kernel (small lattices, site counts that are no multiple of its
64-site chunk), the one-thread-per-site kernel above its limit, both parities
in one launch and one at a time, with and without Naik links, double- and
single-stored links, both precisions, against the oracle.  Tolerance: rounding
of 16 (8) links of 3 complex terms in the stored precision, 1e-14 and 2e-6
relative L2."""
import numpy as np
import pytest

import qopqdp_amd as q
from conftest import MILC

pytestmark = pytest.mark.gpu
EVEN, ODD, EVENODD = 0, 1, 2


@pytest.mark.parametrize("L", [[4, 4, 4, 4], [4, 6, 6, 10], [6, 10, 4, 14], [16, 16, 18, 24], [16, 16, 22, 32]])
@pytest.mark.parametrize("prec", ["D", "F"])
@pytest.mark.parametrize("naik", [True, False])
def test_dslash_matches_oracle(oracle, L, prec, naik):
    U = q.gen_gauge(L, 5100, 0.3)
    oracle.rephase_milc(L, U)
    fat, lng = oracle.make_imp_links(L, U, MILC) if L[0] < 16 else (U, [u[::-1].copy() for u in U])
    if not naik:
        lng = None
    src = q.gen_source(L, 5200, EVENODD)
    if prec == "F":
        src = src.astype(np.float32).astype(np.float64)
    tol = 1e-14 if prec == "D" else 2e-6
    s = q.Session(L)
    fla = s.links_from_raw(fat, lng, prec)
    h = oracle.links(L, fat, lng)
    vin = s.vec(src, EVENODD, prec)
    fn = s.lib.QOP_D3_asqtad_dslash if prec == "D" else s.lib.QOP_F3_asqtad_dslash
    try:
        for st in (1, 0):
            s.set_opts(st=st)
            for eo_out, eo_in in ((EVENODD, EVENODD), (EVEN, ODD), (ODD, EVEN), (EVEN, EVENODD)):
                vout = s.zeros(prec)
                fn(None, fla, 0.07, vout, vin, eo_out, eo_in)
                want = oracle.dslash(h, 0.07, src, eo_out, eo_in)
                got = s.get(vout, EVENODD, prec).astype(np.float64)
                assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want), (st, eo_out, eo_in)
                s.free(vout, prec)
    finally:
        s.set_opts(st=1)
        s.free(vin, prec)
        (s.lib.QOP_D3_asqtad_destroy_L if prec == "D" else s.lib.QOP_F3_asqtad_destroy_L)(fla)
        oracle.free_links(h)
        s.close()
