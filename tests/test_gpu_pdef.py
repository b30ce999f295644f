"""The positive-definite correction visits only tiles whose cells, or whose
neighbours' cells, were marked by the advection kernel: isolated spikes at the
edges of tiles, of a workgroup's levels and of the domain, whose undershoots
reach across those edges, against the oracle bit for bit."""
import numpy as np
import pytest

from common import PROG, case, interior, make_gpu, make_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bc", [1, 2], ids=["periodic", "open"])
@pytest.mark.parametrize("ni,nj,nk", [(8, 9, 8), (64, 8, 17), (65, 10, 16), (130, 13, 9)])
def test_spikes_at_tile_edges(require_gpu, ni, nj, nk, bc):
    cfgd, cols, fields = case(ni=ni, nj=nj, nk=nk, dz=15000.0 / nk, dt=4.0, amp=2.0, seed=ni, bc=bc, npt=3)
    edge = lambda n, w: sorted({c for c in (1, 2, w - 1, w, w + 1, n - 1, n) if 1 <= c <= n})
    spots = [(i, j, k) for i in edge(ni, 64) for j in edge(nj, 4) for k in edge(nk, 8)]
    rng = np.random.default_rng(5)
    # one spike alone, a few, and none at all
    for name, n in (("pta0", 1), ("pta1", 6), ("pta2", 0)):
        fields[name][:] = 0.0 if n else 1.0
        for i, j, k in rng.permutation(spots)[:n]:
            fields[name][k, j + 2, i + 2] = 1.0
    g = make_gpu(cfgd, cols, fields)
    o = make_oracle(cfgd, cols, fields)
    for _ in range(3):
        g.step(1)
        o.step(1)
        for name, stag in PROG + [(f"pta{t}", None) for t in range(3)]:
            a = g.interior(name, stag)
            b = interior(o.f(name), nk, nj, ni, stag)
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), name
    g.close()


@pytest.mark.parametrize("d,ni,nj,nk,sign,hole", [
    # past the periodic seam, domains that end within a tile and on its edge
    ("x", 65, 8, 6, 1, 0), ("x", 100, 9, 6, 1, 0), ("x", 130, 11, 7, 1, 0), ("x", 301, 8, 6, 1, 0),
    ("x", 128, 8, 6, 1, 0), ("x", 65, 8, 6, -1, 64), ("x", 130, 8, 6, -1, 129), ("x", 128, 8, 6, -1, 127),
    # past the edge of a tile's 64 columns
    ("x", 130, 8, 6, 1, 64), ("x", 130, 8, 6, 1, 128), ("x", 130, 8, 6, -1, 63), ("x", 130, 8, 6, -1, 127),
    # the same along y, tiles of 4 rows
    ("y", 8, 9, 6, 1, 0), ("y", 65, 14, 6, 1, 0), ("y", 8, 16, 6, 1, 0), ("y", 65, 14, 6, -1, 13),
    ("y", 65, 14, 6, 1, 8), ("y", 65, 14, 6, -1, 7),
    # one level and two levels a workgroup
    ("z", 65, 9, 20, 1, 10), ("z", 65, 9, 20, -1, 10),
    ("z", 130, 260, 50, 1, 24), ("z", 130, 260, 50, 1, 25), ("z", 130, 260, 50, -1, 24), ("z", 130, 260, 50, -1, 25),
])
def test_undershoot_paid_across_an_edge(require_gpu, d, ni, nj, nk, sign, hole):
    """A sharp front along d in a constant mass flux, all else at rest: ahead
    of it the fifth-order flux leaves one cell negative (index hole, from 0),
    and the cell between the front and it, on the other side of the edge, pays
    for it although nothing in its own tile is marked."""
    import ctypes as C

    import pyoracle
    from cm1_amd import _native as N

    cfgd, cols, fields = case(ni=ni, nj=nj, nk=nk, dz=15000.0 / nk, dt=4.0, bc=1)
    g = make_gpu(cfgd, cols, fields)
    o = make_oracle(cfgd, cols, fields)
    n, axis = {"x": (ni, 2), "y": (nj, 1), "z": (nk, 0)}[d]
    pay = (hole - sign) % n
    # 1 behind the front over more than a tile, so that its rear end, where the
    # flux undershoots as well, is in another one where the domain has one
    s = np.zeros(n, np.float32)
    s[(hole - sign * np.arange(2, 2 + min(n - 6, 76 if d == "x" else 6))) % n] = 1.0
    k, j, i = slice(1, nk + 1), slice(3, nj + 3), slice(3, ni + 3)
    for name in ("q3d2", "qa2", "qten2", "divx", "rru", "rrv", "rrw"):
        o.f(name)[:] = 0.0
    for name in ("q3d2", "qa2"):
        o.f(name)[k, j, i] = s.reshape([n if a == axis else 1 for a in range(3)])
        o.L.cm1o_bc(o.h, pyoracle.FID[name], 0)
    if d == "z":
        o.f("rrw")[2:nk + 1] = sign * 5.0
    else:
        o.f("rru" if d == "x" else "rrv")[:] = sign * 20.0
    for name in ("q3d2", "qa2", "qten2", "divx", "rru", "rrv", "rrw"):
        g.put(name, np.ascontiguousarray(o.f(name)))

    def oracle(pdef):
        o.f("qten2")[:] = 0.0
        o.L.cm1o_advs(o.h, 3, pyoracle.FID["q3d2"], pyoracle.FID["qa2"], pyoracle.FID["qten2"], pdef, pdef,
                      C.c_double(1.0e-20))
        return o.f("qten2")[k, j, i].copy()

    plain, fixed = oracle(0), oracle(1)
    # the case is the one meant: `hole` alone is negative near the front, and
    # the correction takes from `pay` (every column, row and level of them)
    new = np.moveaxis(o.f("qa2")[k, j, i] + np.float32(cfgd["dt"]) * plain, axis, 0).reshape(n, -1)
    assert (new[hole] < 0.0).all() and (new[pay] > 0.0).all()
    if d == "x" and not (ni == 65 and sign < 0):
        own = [q for q in range(n) if q // 64 == pay // 64 and q != hole]
        assert not (new[own] < 0.0).any()
    assert (np.moveaxis(plain != fixed, axis, 0).reshape(n, -1)[pay]).all()
    N.check(g.L.cm1g_advs(g.h, 3, N.FID["q3d2"], N.FID["qa2"], N.FID["qten2"], 1, 1, C.c_float(cfgd["dt"]),
                          C.c_double(1.0e-20)), "cm1g_advs")
    a = np.ascontiguousarray(g.get("qten2")[k, j, i])
    assert np.array_equal(a.view(np.uint32), fixed.view(np.uint32))
    g.close()


@pytest.mark.parametrize("u", [20.0, -20.0], ids=["up", "down"])
@pytest.mark.parametrize("ni", [65, 130, 301])
def test_step_across_the_periodic_seam(require_gpu, ni, u):
    """The whole step in a calm cross flow: a tracer that ends sharply at the
    seam, uniform wind, no other motion, so nothing else marks a tile."""
    nj, nk = 9, 8
    cfgd, cols, fields = case(ni=ni, nj=nj, nk=nk, dz=15000.0 / nk, dt=4.0, bc=1, amp=0.0, umax=0.0, noise=0.0, npt=1)
    fields["ua"][:] = u
    if "u0" in cols:
        cols["u0"][:] = u
    s = np.zeros(ni, np.float32)
    s[(np.arange(2, 2 + min(ni - 6, 76)) * (-1 if u > 0 else 1) - (u < 0)) % ni] = 1.0
    fields["pta0"][:] = 0.0
    fields["pta0"][1:nk + 1, 3:nj + 3, 3:ni + 3] = s

    def oracle(pdtra):
        o = make_oracle(dict(cfgd, pdtra=pdtra), cols, fields)
        o.step(1)
        return interior(o.f("pta0"), nk, nj, ni).copy()

    plain, fixed = oracle(0), oracle(1)
    pay = ni - 1 if u > 0 else 0
    assert (plain[:, :, pay] != fixed[:, :, pay]).all()
    g = make_gpu(cfgd, cols, fields)
    g.step(1)
    a = g.interior("pta0")
    assert np.array_equal(a.view(np.uint32), fixed.view(np.uint32))
    g.close()
