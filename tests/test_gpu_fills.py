"""Halo fills from interior points in one pass (cm1g_bc) against the oracle's
two passes over an array, whole boxes equal, and the reductions that end a stage
(dry mass, Courant number, radiation speeds, rain budget) at sizes around
their workgroups' chunks, against the oracle."""
import numpy as np
import pytest

import pyoracle
from cm1_amd import _native as N
from common import PROG, case, interior, make_gpu, make_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("we,sn", [(1, 1), (2, 2), (1, 2), (2, 1)], ids=["periodic", "open", "we-periodic", "sn-periodic"])
@pytest.mark.parametrize("ni,nj,nk", [(8, 8, 6), (37, 130, 9), (260, 11, 7)])
def test_fill_equals_two_passes(require_gpu, ni, nj, nk, we, sn):
    cfgd, cols, fields = case(ni=ni, nj=nj, nk=nk)
    cfgd.update(wbc=we, ebc=we, sbc=sn, nbc=sn)
    g = make_gpu(cfgd, cols, fields)
    o = make_oracle(cfgd, cols, fields)
    rng = np.random.default_rng(ni + nk)
    for name, kind in N.BC.items():
        a = rng.standard_normal((nk + 3, nj + 7, ni + 7)).astype(np.float32)
        o.f("dum3")[:] = a
        g.put("dum3", a)
        N.check(g.L.cm1g_bc(g.h, N.FID["dum3"], kind), "cm1g_bc")
        o.L.cm1o_bc(o.h, pyoracle.FID["dum3"], kind)
        assert np.array_equal(g.get("dum3"), o.f("dum3")), name
    g.close()


@pytest.mark.parametrize("ni,nj,nk", [(8, 33, 6), (129, 8, 64), (65, 40, 65), (8, 8, 300)])
def test_stage_reductions_match_oracle(require_gpu, ni, nj, nk):
    cfgd, cols, fields = case(ni=ni, nj=nj, nk=nk, dz=15000.0 / nk, dt=2.0, amp=3.0)
    k, j, i = slice(1, nk + 1), slice(3, nj + 3), slice(3, ni + 3)
    fields["qa2"][k, j, i] = 2.0e-3 * (cols["zh"][k, None, None] < 4000.0)  # rain, so that the budget counts
    g = make_gpu(cfgd, cols, fields)
    o = make_oracle(cfgd, cols, fields)
    cfl = g.step(2)
    o.step(2)
    for name, stag in PROG:
        a, b = g.interior(name, stag), interior(o.f(name), nk, nj, ni, stag)
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), name
    # the rain budget adds rows in i order, then the rows: the oracle's order
    s, t = g.scalars(), o.scalars()
    assert s["train"] == t["train"] > 0.0
    assert cfl == s["cflmax"] == np.float32(t["cflmax"]) > 0.0
    g.close()
