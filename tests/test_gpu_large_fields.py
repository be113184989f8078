"""Link construction and forces on a lattice whose matrix fields (413 MB) are
larger than the blocks the allocator keeps, where a call's workspace is one
allocation.  The fields repeat those of a small lattice, so the results repeat
the small lattice's: relative L2 <= 1e-13, the rounding of the sums per site,
which do not depend on the volume."""
import ctypes as C

import numpy as np
import pytest

import qopqdp_amd as q

pytestmark = pytest.mark.gpu
SMALL, LARGE = [4, 4, 8, 14], [32, 32, 40, 70]
P = C.c_void_p


def results(L, U, xs, where):
    """Asqtad and HISQ force of the terms xs and a Dslash on the asqtad links,
    at the raw sites `where`."""
    s = q.Session(L)
    zero = np.zeros((s.V, 3, 3, 2))
    try:
        g = s.gauge(U)
        vs = [s.vec(x) for x in xs]
        n = len(vs)
        eps = (C.c_double * n)(*[0.3 / (1 + k) for k in range(n)])
        c, hc, info = q.QOPAsqtadCoeffs(**q.MILC_ASQTAD), q.hisq_coeffs(), q.QOPInfo()
        out = []
        for hisq in (False, True):
            f = s.force([zero] * 4)
            if hisq:
                h = s.lib.QOP_D3_hisq_create_L_from_G(C.byref(info), C.byref(hc), g)
                s.lib.QOP_D3_hisq_force_multi(C.byref(info), h, f, C.byref(hc), eps, (P * n)(*vs), (C.c_int * 1)(n))
                s.lib.QOP_D3_hisq_destroy_L(h)
            else:
                s.lib.QOP_D3_asqtad_force_multi(C.byref(info), g, f, C.byref(c), eps, (P * n)(*vs), n)
            assert info.status == 0
            out += [x[where].copy() for x in s.get_force(f)]
            s.lib.QOP_D3_destroy_F(f)
        fla, _ = s.links_from_gauge(g)
        v = s.zeros()
        s.lib.QOP_D3_asqtad_dslash(None, fla, 0.1, v, vs[0], 2, 2)
        out.append(s.get(v)[where].copy())
        s.lib.QOP_D3_asqtad_destroy_L(fla)
        for x in vs + [v]:
            s.free(x)
        s.lib.QOP_D3_destroy_G(g)
        return out
    finally:
        s.close()


def test_workspace_in_one_allocation():
    U = q.gen_gauge(SMALL, 8000, 0.3)
    xs = [q.gen_source(SMALL, 8100 + k, 2) for k in range(2)]
    x = q.raw_coords_all(LARGE) % np.array(SMALL)
    lex = ((x[:, 0] * SMALL[1] + x[:, 1]) * SMALL[2] + x[:, 2]) * SMALL[3] + x[:, 3]
    V = int(np.prod(SMALL))
    tile = np.where(x.sum(axis=1) & 1, (lex + V) // 2, lex // 2)
    del x, lex
    rng = np.random.default_rng(5)
    where = rng.choice(tile.size, 20000, replace=False)
    where[:2] = 0, tile.size - 1
    want = results(SMALL, U, xs, slice(None))
    got = results(LARGE, [u[tile] for u in U], [v[tile] for v in xs], where)
    for a, b in zip(got, want):
        b = b[tile[where]]
        assert np.linalg.norm(a - b) <= 1e-13 * np.linalg.norm(b)
