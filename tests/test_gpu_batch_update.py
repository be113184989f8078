"""Reliable updates of the batched solver at the edges of their launches:
lattices smaller than a block and with a partial 64-site chunk, with and
without Naik links, both sloppy precisions, one slot to more systems than
slots, and a lattice above the limit where the increments are folded in a pass
of their own.  Every system reaches its FP64 true residual, recomputed here
with the FP64 operator, and its bits do not depend on its batch."""
import ctypes as C

import numpy as np
import pytest

import qopqdp_amd as q
from conftest import MILC

pytestmark = pytest.mark.gpu
EVEN, ODD, EVENODD = 0, 1, 2
P = C.c_void_p


def batch(s, fla, m, tol, srcs, eo, capacity, prec):
    n = len(srcs)
    vin, vout = [s.vec(x) for x in srcs], [s.zeros() for _ in srcs]
    ras = [q.resid_arg_default() for _ in srcs]
    for r in ras:
        r.rsqmin = tol * tol
    ia, info = q.invert_arg_default(), q.QOPInfo()
    ia.evenodd, ia.max_iter = eo, 5000
    rc = s.lib.QOPX_D3_asqtad_invert_batch(
        C.byref(info), fla, C.byref(ia), (P * n)(*[C.addressof(r) for r in ras]), (C.c_double * n)(*([m] * n)),
        (P * n)(*vout), (P * n)(*vin), n, capacity, prec, None)
    assert rc == n and info.status == 0
    out = [s.get(v) for v in vout]
    for v in vin + vout:
        s.free(v)
    return out


def residual(s, fla, m, x, src, eo):
    """|src - A x / m| / |src| with the library's FP64 Dslash."""
    v, t, o = s.vec(x), s.zeros(), s.zeros()
    s.lib.QOP_D3_asqtad_dslash(None, fla, 0.0, t, v, 1 - eo, eo)
    s.lib.QOP_D3_asqtad_dslash(None, fla, 0.0, o, t, eo, 1 - eo)
    half = slice(0, s.V // 2) if eo == EVEN else slice(s.V // 2, s.V)
    r = src[half] - (m * m * x[half] - s.get(o)[half]) / m
    for h in (v, t, o):
        s.free(h)
    return np.linalg.norm(r) / np.linalg.norm(src[half])


@pytest.mark.parametrize("L,n,capacity,eo", [([4, 4, 4, 4], 1, 1, EVEN), ([6, 4, 6, 10], 5, 3, ODD),
                                             ([4, 6, 4, 10], 9, 9, EVEN), ([16, 16, 32, 34], 3, 2, EVEN)])
@pytest.mark.parametrize("naik", [True, False])
@pytest.mark.parametrize("prec", [16, 32])
def test_reliable_updates(oracle, L, n, capacity, eo, naik, prec):
    m, tol = 0.3, 1e-10
    U = q.gen_gauge(L, 6100, 0.3)
    oracle.rephase_milc(L, U)
    s = q.Session(L)
    g = s.gauge(U)
    fla, _ = s.links_from_gauge(g, MILC if naik else dict(MILC, naik=0.0))
    try:
        srcs = [q.gen_source(L, 6200 + i, eo) for i in range(n)]
        out = batch(s, fla, m, tol, srcs, eo, capacity, prec)
        for x, b in zip(out, srcs):
            assert residual(s, fla, m, x, b, eo) <= 1.01 * tol
        alone = batch(s, fla, m, tol, srcs[-1:], eo, 1, prec)[0]
        assert np.array_equal(alone, out[-1])
    finally:
        s.lib.QOP_D3_asqtad_destroy_L(fla)
        s.lib.QOP_D3_destroy_G(g)
        s.close()
