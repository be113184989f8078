"""Solves on the library stream while a request server creates and evicts its
batches from its own thread: neither side's iteration graphs hold or disturb
the other's work, so every result has the bits it has alone, on both sides."""
import ctypes as C
import threading

import numpy as np
import pytest

import qopqdp_amd as q
from conftest import MILC

pytestmark = pytest.mark.gpu
EVEN, EVENODD = 0, 2
L = [4, 4, 6, 8]


def solve(s, fla, src, eo):
    ia, ra, info = q.invert_arg_default(), q.resid_arg_default(), q.QOPInfo()
    ia.evenodd, ra.rsqmin = eo, 1e-18
    vin, vout = s.vec(src, EVENODD), s.zeros()
    s.lib.QOP_D3_asqtad_invert(C.byref(info), fla, C.byref(ia), C.byref(ra), 0.1, vout, vin)
    assert info.status == 0
    out = s.get(vout)
    s.free(vin)
    s.free(vout)
    return out


def test_solves_beside_a_server_that_rebuilds_its_batches():
    U = [q.gen_gauge(L, 7000 + k, 0.3) for k in range(3)]
    srcs = [q.gen_source(L, 7100 + i, EVEN) for i in range(2)]

    def make_server(**kw):
        srv = q.Server(capacity=2, prec=32, **kw)
        for k in range(2):
            srv.add_gauge(L, U[k], MILC)
        return srv

    def ask(srv, i):
        out, st, _, _ = srv.wait(srv.submit(i % 2, srcs[i % 2], 0.1, 1e-9, EVEN))
        assert st == 0
        return out

    srv = make_server()
    used = srv.stats()["bytes_used"]
    want_srv = [ask(srv, i) for i in range(2)]
    one = (srv.stats()["bytes_used"] - used) / 2
    srv.close()

    s = q.Session(L)
    g = s.gauge(U[2])
    fla, _ = s.links_from_gauge(g)
    full = q.gen_source(L, 7200, EVENODD)
    want = {eo: solve(s, fla, full, eo) for eo in (EVEN, EVENODD)}
    srv = make_server(max_bytes=int(used + 1.5 * one))  # one batch at a time
    errors, asked = [], [0]
    stop = threading.Event()

    def feed():
        try:
            while not stop.is_set():
                i = asked[0]
                if not np.array_equal(ask(srv, i), want_srv[i % 2]):
                    errors.append(i)
                asked[0] += 1
        except Exception as e:  # noqa: BLE001 - reported by the main thread
            errors.append(e)

    t = threading.Thread(target=feed)
    t.start()
    try:
        for k in range(200):
            eo = EVENODD if k % 2 else EVEN
            assert np.array_equal(solve(s, fla, full, eo), want[eo]), k
            if errors or (k >= 60 and asked[0] >= 20):
                break
    finally:
        stop.set()
        t.join()
        srv.close()
        s.lib.QOP_D3_asqtad_destroy_L(fla)
        s.lib.QOP_D3_destroy_G(g)
        s.close()
    assert not errors and asked[0] >= 4


def test_solves_beside_a_server_of_the_reference_algorithm():
    """A server of precision 64 solves on the library stream too: its worker's
    reductions are its own."""
    U = [q.gen_gauge(L, 7300 + k, 0.3) for k in range(2)]
    src = q.gen_source(L, 7400, EVEN)
    srv = q.Server(capacity=1, prec=64)
    srv.add_gauge(L, U[0], MILC)

    def ask():
        out, st, res, _ = srv.wait(srv.submit(0, src, 0.1, 1e-9, EVEN))
        assert st == 0
        return out

    want_srv = ask()
    s = q.Session(L)
    g = s.gauge(U[1])
    fla, _ = s.links_from_gauge(g)
    full = q.gen_source(L, 7500, EVENODD)
    want = {eo: solve(s, fla, full, eo) for eo in (EVEN, EVENODD)}
    errors, asked = [], [0]
    stop = threading.Event()

    def feed():
        try:
            while not stop.is_set():
                if not np.array_equal(ask(), want_srv):
                    errors.append(asked[0])
                asked[0] += 1
        except Exception as e:  # noqa: BLE001 - reported by the main thread
            errors.append(e)

    t = threading.Thread(target=feed)
    t.start()
    try:
        for k in range(100):
            eo = EVENODD if k % 2 else EVEN
            assert np.array_equal(solve(s, fla, full, eo), want[eo]), k
            if errors or (k >= 40 and asked[0] >= 20):
                break
    finally:
        stop.set()
        t.join()
        srv.close()
        s.lib.QOP_D3_asqtad_destroy_L(fla)
        s.lib.QOP_D3_destroy_G(g)
        s.close()
    assert not errors and asked[0] >= 4
