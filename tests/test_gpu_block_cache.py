"""The block cache behind device allocations: results do not depend on what a
reused block held, a link object reloaded on another lattice gets an array of
that lattice, several threads may allocate and free (their calls here wait for
their own work; blocks freed with work in flight are the host checks' and
test_gpu_beside_server's), freed blocks are kept, and QOP_finalize gives them
back."""
import ctypes as C
import threading

import numpy as np
import pytest

import qopqdp_amd as q

pytestmark = pytest.mark.gpu
EVEN, EVENODD = 0, 2


def free_bytes():
    hip = C.CDLL("libamdhip64.so")
    fr, tot = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(fr), C.byref(tot)) == 0
    return fr.value


def solve(s, fla, src, eo):
    ia, ra, info = q.invert_arg_default(), q.resid_arg_default(), q.QOPInfo()
    ia.evenodd = eo
    ra.rsqmin = 1e-16
    vin, vout = s.vec(src), s.zeros()
    s.lib.QOP_D3_asqtad_invert(C.byref(info), fla, C.byref(ia), C.byref(ra), 0.2, vout, vin)
    out = s.get(vout)
    s.free(vin)
    s.free(vout)
    return out


def load(s, fla, g):
    c, info = q.QOPAsqtadCoeffs(**q.MILC_ASQTAD), q.QOPInfo()
    s.lib.QOP_D3_asqtad_load_L_from_G(C.byref(info), fla, C.byref(c), g)
    assert info.status == 0


@pytest.mark.parametrize("first,second", [([4, 4, 4, 8], [6, 8, 4, 10]), ([8, 8, 8, 8], [4, 4, 4, 4]),
                                          ([4, 8, 4, 8], [8, 4, 8, 4])])
def test_reloaded_links_and_repeated_solves(first, second):
    s = q.Session(first)
    g = s.gauge(q.gen_gauge(first, 31, 0.3))
    fla, _ = s.links_from_gauge(g)
    a = solve(s, fla, q.gen_source(first, 32, EVENODD), EVENODD)
    load(s, fla, g)  # in place
    b = solve(s, fla, q.gen_source(first, 32, EVENODD), EVENODD)
    assert np.array_equal(a, b)
    s.lib.QOP_D3_destroy_G(g)
    s.close()
    s = q.Session(second)
    try:
        g = s.gauge(q.gen_gauge(second, 33, 0.3))
        load(s, fla, g)  # the object moves to another lattice
        fresh, _ = s.links_from_gauge(g)
        src = q.gen_source(second, 34, EVEN)
        want = solve(s, fresh, src, EVEN)
        for _ in range(3):
            assert np.array_equal(solve(s, fla, src, EVEN), want)
        for x in (fla, fresh):
            s.lib.QOP_D3_asqtad_destroy_L(x)
        s.lib.QOP_D3_destroy_G(g)
    finally:
        s.close()


def test_threads_and_finalize():
    L = [8, 8, 8, 8]
    s = q.Session(L)
    src = [q.gen_source(L, 40 + i, EVENODD) for i in range(4)]
    before = free_bytes()
    errors = []

    def work(i):
        for _ in range(20):
            v = s.vec(src[i])
            if not np.array_equal(s.get(v), src[i]):
                errors.append(i)
            s.free(v)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors
    s.close()
    assert free_bytes() >= before - (16 << 20)  # reduction scratch may stay


def test_freed_blocks_are_kept_until_finalize():
    L = [16, 16, 16, 32]  # a vector is 6.3 MB
    s = q.Session(L)
    s.free(s.zeros())
    before = free_bytes()
    vs = [s.zeros() for _ in range(60)]
    held = free_bytes()
    assert held <= before - (350 << 20)
    for v in vs:
        s.free(v)
    assert free_bytes() <= held + (16 << 20)
    vs = [s.zeros() for _ in range(60)]  # from the kept blocks
    assert free_bytes() >= held - (16 << 20)
    for v in vs:
        s.free(v)
    s.close()
    assert free_bytes() >= before - (16 << 20)
