"""Link construction where device memory is short.  A 32^3x64 configuration
whose links and workspace (28 fields of 302 MB beside the gauge field) do not
fit in what is left, while the links and the raw links (24) do, gets the same
links as with memory to spare.  Where no way fits, the request server refuses
the configuration and all it had taken is free again."""
import ctypes as C

import numpy as np
import pytest

import qopqdp_amd as q

pytestmark = pytest.mark.gpu
L = [32, 32, 32, 64]
FIELD = 32 * 32 * 32 * 64 * 144


class Ballast:
    """Device memory held so that `left` bytes are free."""

    def __init__(self, left):
        self.hip, self.held = C.CDLL("libamdhip64.so"), []
        fr, tot = C.c_size_t(), C.c_size_t()
        for size in (16 << 30, 1 << 30, 64 << 20):
            while True:
                assert self.hip.hipMemGetInfo(C.byref(fr), C.byref(tot)) == 0
                p = C.c_void_p()
                if fr.value < left + size or self.hip.hipMalloc(C.byref(p), C.c_size_t(size)) != 0:
                    break
                self.held.append(p)
        assert left <= fr.value < left + (128 << 20)

    def free(self):
        fr, tot = C.c_size_t(), C.c_size_t()
        assert self.hip.hipMemGetInfo(C.byref(fr), C.byref(tot)) == 0
        return fr.value

    def drop(self):
        for p in self.held:
            assert self.hip.hipFree(p) == 0


def dslash(s, fla, vec):
    out = s.zeros()
    s.lib.QOP_D3_asqtad_dslash(None, fla, 0.1, out, vec, 2, 2)
    r = s.get(out)
    s.free(out)
    return r


def test_links_where_the_direct_way_does_not_fit():
    s = q.Session(L)
    g = s.gauge(q.gen_gauge(L, 9000, 0.3))
    src = s.vec(q.gen_source(L, 9001, 2))
    fla, _ = s.links_from_gauge(g)
    want = dslash(s, fla, src)
    s.lib.QOP_D3_asqtad_destroy_L(fla)
    s.close()  # kept blocks go back
    s = q.Session(L)
    ballast = Ballast(int(25.5 * FIELD))
    try:
        c, info = q.QOPAsqtadCoeffs(**q.MILC_ASQTAD), q.QOPInfo()
        fla = s.lib.QOP_D3_asqtad_create_L_from_G(C.byref(info), C.byref(c), g)
        assert fla and info.status == 0
        got = dslash(s, fla, src)
        s.lib.QOP_D3_asqtad_destroy_L(fla)
    finally:
        ballast.drop()
        s.free(src)
        s.lib.QOP_D3_destroy_G(g)
        s.close()
    assert np.array_equal(got, want)


def test_a_refused_configuration_leaves_nothing_behind():
    U = q.gen_gauge(L, 9002, 0.3)
    srv = q.Server(capacity=1, prec=32, max_bytes=1 << 40)
    ballast = Ballast(20 * FIELD)
    try:
        before = ballast.free()
        with pytest.raises(RuntimeError):
            srv.add_gauge(L, U)
        assert ballast.free() >= before - (64 << 20)
        assert srv.stats()["bytes_used"] == 0
    finally:
        ballast.drop()
        srv.close()
