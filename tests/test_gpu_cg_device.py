"""The device iterations of the reference CG and multi-shift CG at the edges of
their launches: lattices smaller than a block, whose site count is no multiple
of the 64-site reduction chunk or of a block, odd iteration chunks, restarts
inside a solve, the relative-residual test, single-stored links and both
precisions, against the oracle's solves.

Tolerance: both solutions have relative residual <= tol, so they differ by at
most 2 tol kappa with kappa = (m^2 + 8) / m^2 bounding the condition number of
A = m^2 - D_eo D_oe on these links.  Where the relative-residual test stops the
solve the two are iterates of the same number: a change of 1e-13 in the source
moves the oracle's by 2e-13 and its iteration count and reported residuals not
at all (8 digits), so 1e-9, the same count and 4 digits are asked for.
"""
import ctypes as C

import numpy as np
import pytest

import qopqdp_amd as q
from conftest import MILC

pytestmark = pytest.mark.gpu
EVEN, ODD, EVENODD = 0, 1, 2
M = 0.3
KAPPA = (M * M + 8.0) / (M * M)


@pytest.mark.parametrize("L", [[4, 4, 4, 4], [4, 6, 4, 6], [6, 10, 4, 14], [8, 4, 6, 12]])
@pytest.mark.parametrize("prec,eo,restart,relmin,opts", [
    ("D", EVENODD, 1000, 0.0, {}),
    ("D", EVENODD, 9, 0.0, dict(qmx_chunk=5)),
    ("D", EVENODD, 1000, 1e-12, {}),
    ("D", EVEN, 1000, 1e-12, {}),
    ("D", ODD, 1000, 0.0, dict(qmx_chunk=1)),
    ("D", EVENODD, 1000, 0.0, dict(st=0)),
    ("D", EVEN, 1000, 0.0, dict(qmx_graph=0)),
    ("F", EVENODD, 1000, 0.0, {}),
    ("F", EVEN, 1000, 0.0, {}),
])
def test_solve_matches_oracle(oracle, L, prec, eo, restart, relmin, opts):
    tol = 1e-8 if prec == "D" else 1e-4
    U = q.gen_gauge(L, 4100, 0.3)
    oracle.rephase_milc(L, U)
    fat, lng = oracle.make_imp_links(L, U, MILC)
    src = q.gen_source(L, 4200, eo)
    s = q.Session(L)
    fla = s.links_from_raw(fat, lng, prec)
    h = oracle.links(L, fat, lng)
    vin, vout = s.vec(src, EVENODD, prec), s.zeros(prec)
    try:
        s.set_opts(st=1, qmx_chunk=16, qmx_graph=1)
        if opts:
            s.set_opts(**opts)
        ia, ra, info = q.invert_arg_default(), q.resid_arg_default(), q.QOPInfo()
        ia.evenodd, ia.restart, ia.max_restarts = eo, restart, 60
        ra.rsqmin, ra.relmin = tol * tol, relmin
        fn = s.lib.QOP_D3_asqtad_invert if prec == "D" else s.lib.QOP_F3_asqtad_invert
        fn(C.byref(info), fla, C.byref(ia), C.byref(ra), M, vout, vin)
        assert info.status == 0
        out = s.get(vout, EVENODD, prec).astype(np.float64)
        want, ora, _ = oracle.invert(h, M, src, eo, tol * tol, restart=restart, max_restarts=60, relmin=relmin)
        sl = {EVEN: slice(0, s.V // 2), ODD: slice(s.V // 2, s.V), EVENODD: slice(0, s.V)}[eo]
        d = np.linalg.norm(out[sl] - want[sl]) / np.linalg.norm(want[sl])
        if relmin == 0:
            assert d <= 2 * tol * KAPPA
            if prec == "D":
                assert abs(ra.final_iter - ora.final_iter) <= max(2, 0.02 * ora.final_iter)
        else:
            assert d <= 1e-9
            assert abs(ra.final_iter - ora.final_iter) <= 1
            assert ra.final_rel <= relmin
            assert ra.final_rel == pytest.approx(ora.final_rel, rel=1e-4)
            assert ra.final_rsq == pytest.approx(ora.final_rsq, rel=1e-4)
            if eo == EVEN:  # it is the relative residual that stops it, before the other would
                _, plain, _ = oracle.invert(h, M, src, eo, tol * tol, restart=restart, max_restarts=60)
                assert ra.final_iter < plain.final_iter
    finally:
        s.set_opts(st=1, qmx_chunk=16, qmx_graph=1)
        s.free(vin, prec)
        s.free(vout, prec)
        (s.lib.QOP_D3_asqtad_destroy_L if prec == "D" else s.lib.QOP_F3_asqtad_destroy_L)(fla)
        oracle.free_links(h)
        s.close()


@pytest.mark.parametrize("L", [[4, 4, 4, 4], [4, 6, 4, 6], [6, 10, 4, 14], [8, 4, 6, 12]])
@pytest.mark.parametrize("eo", [EVEN, ODD])
@pytest.mark.parametrize("rsqmin,relmin,opts", [
    (1e-16, 0.0, {}),
    (1e-16, 0.0, dict(qmx_chunk=1)),
    (1e-16, 0.0, dict(qmx_chunk=5)),
    (1e-16, 0.0, dict(qmx_graph=0)),
    (1e-16, 0.0, dict(st=0)),
    (1e-16, 1e-12, dict(qmx_chunk=5)),
    (1e-8, 1e-12, {}),
])
def test_multi_shift_matches_oracle(oracle, L, eo, rsqmin, relmin, opts):
    """Three masses in one solve.  The two larger lattices pass the host's check
    at iteration 100 (105 to 114 iterations) and go on after it; with relmin the
    x and p updates are separate passes, and where rsqmin is the tighter of the
    two the reference's refinement runs on (up to 443 iterations).  The oracle's
    solutions move by 2e-13 for a change of 1e-13 in the source, its iteration
    counts not at all: 1e-9 and one iteration."""
    masses = [0.05, 0.1, 0.3]
    n = len(masses)
    U = q.gen_gauge(L, 4100, 0.3)
    oracle.rephase_milc(L, U)
    fat, lng = oracle.make_imp_links(L, U, MILC)
    src = q.gen_source(L, 4200, eo)
    s = q.Session(L)
    fla = s.links_from_raw(fat, lng)
    h = oracle.links(L, fat, lng)
    vin, vouts = s.vec(src), [s.zeros() for _ in masses]
    try:
        s.set_opts(st=1, qmx_chunk=16, qmx_graph=1)
        if opts:
            s.set_opts(**opts)
        ia, info = q.invert_arg_default(), q.QOPInfo()
        ia.evenodd, ia.max_restarts = eo, 5
        ras = [q.resid_arg_default() for _ in masses]
        for r in ras:
            r.rsqmin, r.relmin = rsqmin, relmin
        m = (C.c_double * n)(*masses)
        rp = (C.POINTER(q.QOPResidArg) * n)(*[C.pointer(r) for r in ras])
        op = (C.c_void_p * n)(*vouts)
        s.lib.QOP_D3_asqtad_invert_multi(
            C.byref(info), fla, C.byref(ia), (C.c_void_p * 1)(C.addressof(rp)), (C.c_void_p * 1)(C.addressof(m)),
            (C.c_int * 1)(n), (C.c_void_p * 1)(C.addressof(op)), (C.c_void_p * 1)(vin), 1)
        assert info.status == 0
        want, oras, _ = oracle.invert_multi(h, [masses], [src], eo, rsqmin, max_restarts=5, relmin=relmin)
        sl = slice(0, s.V // 2) if eo == EVEN else slice(s.V // 2, s.V)
        for v, w, ra, ora in zip(vouts, want, ras, oras):
            d = np.linalg.norm(s.get(v)[sl] - w[sl]) / np.linalg.norm(w[sl])
            assert d <= 1e-9
            assert abs(ra.final_iter - ora.final_iter) <= 1
            if relmin > 0:
                assert ra.final_rsq == pytest.approx(ora.final_rsq, rel=1e-4)
                assert ra.final_rel == pytest.approx(ora.final_rel, rel=1e-4)
            else:
                assert ra.final_rsq <= rsqmin
    finally:
        s.set_opts(st=1, qmx_chunk=16, qmx_graph=1)
        s.free(vin)
        for v in vouts:
            s.free(v)
        s.lib.QOP_D3_asqtad_destroy_L(fla)
        oracle.free_links(h)
        s.close()
