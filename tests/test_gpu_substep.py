"""The acoustic substep's kernels at the edges of their tiles (64 columns, 4,
8 or 12 levels per wavefront, 64, 96 or 192 levels per workgroup) and of the
averages' pairing of substeps, against the oracle bit for bit."""
import numpy as np
import pytest

from common import PROG, case, interior, make_gpu, make_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ni,nj,nk,nsound,bc", [
    (8, 8, 6, 2, 2),        # the smallest grid; single-substep stages
    (65, 9, 64, 4, 2),      # one column past a tile, every level of the 4-level form
    (63, 8, 61, 6, 1),      # a last wavefront with one level
    (64, 1025, 17, 6, 2),   # 8 levels per wavefront
    (130, 520, 64, 6, 1),   # the same, full, three tiles per row
    (12, 10, 65, 6, 2),     # 12 levels per wavefront, the last one short
    (70, 8, 96, 8, 1),      # full
    (9, 8, 97, 6, 2),       # sixteen wavefronts
    (8, 9, 192, 4, 1),      # full
    (8, 8, 193, 6, 2),      # one thread per column
])
def test_substep_edges_match_oracle(require_gpu, ni, nj, nk, nsound, bc):
    dz = 15000.0 / nk
    cfgd, cols, fields = case(ni=ni, nj=nj, nk=nk, nsound=nsound, bc=bc, dz=dz, dt=0.4 * nsound, amp=2.0)
    g = make_gpu(cfgd, cols, fields)
    o = make_oracle(cfgd, cols, fields)
    for n in (1, 2):  # the first step and one that starts from exchanged buffers
        g.step(n)
        o.step(n)
        for name, stag in PROG + [("ppx", None)]:
            a = g.interior(name, stag)
            b = interior(o.f(name), nk, nj, ni, stag)
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (n, name)
    g.close()


@pytest.mark.parametrize("ni,nj,nk,nsound,bc", [
    (64, 2047, 7, 4, 1),    # slabs, one tile short of the line
    (64, 2048, 7, 4, 2),    # one thread per column
    (65, 1024, 6, 2, 1),    # the fewest levels, single-substep stages
    (64, 2048, 12, 6, 1),
    (64, 2048, 13, 6, 2),   # slabs
    (130, 1279, 20, 6, 1),  # slabs, three tiles short of the second line
    (130, 1280, 20, 6, 2),  # one thread per column
    (130, 1280, 21, 4, 1),  # slabs
])
def test_shallow_wide_grids_match_oracle(require_gpu, ni, nj, nk, nsound, bc):
    """Either side of the rule that sends shallow columns of wide grids to the
    one-thread-per-column kernel."""
    cfgd, cols, fields = case(ni=ni, nj=nj, nk=nk, nsound=nsound, bc=bc, dz=15000.0 / nk, dt=0.4 * nsound, amp=2.0)
    g = make_gpu(cfgd, cols, fields)
    o = make_oracle(cfgd, cols, fields)
    for n in (1, 1):  # the first step and one that starts from exchanged buffers
        g.step(n)
        o.step(n)
        for name, stag in PROG + [("ppx", None)]:
            a = g.interior(name, stag)
            b = interior(o.f(name), nk, nj, ni, stag)
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), name
    g.close()


@pytest.mark.parametrize("ni,nj,nk,nsound,bc", [
    (8, 8, 6, 2, 2),       # single-substep stages
    (9, 8, 7, 5, 2),       # an odd count
    (65, 9, 30, 7, 1),
    (130, 12, 13, 10, 2),
    (12, 10, 49, 12, 1),
])
@pytest.mark.parametrize("held", [False, True], ids=["exchanged", "addresses-held"])
def test_explicit_substep_matches_oracle(require_gpu, ni, nj, nk, nsound, bc, held):
    """psolver 2; also with the address of ua handed out, when every stage
    starts from the 3-D arrays themselves."""
    import ctypes as C
    from cm1_amd import _native as N
    cfgd, cols, fields = case(ni=ni, nj=nj, nk=nk, nsound=nsound, bc=bc, dz=15000.0 / nk, dt=0.25 * nsound, amp=2.0,
                              psolver=2)
    g = make_gpu(cfgd, cols, fields)
    o = make_oracle(cfgd, cols, fields)
    if held:
        p = C.c_void_p()
        N.check(g.L.cm1g_field_ptr(g.h, N.FID["ua"], C.byref(p)), "cm1g_field_ptr")
    for n in (1, 2):
        g.step(n)
        o.step(n)
        for name, stag in PROG + [("ppx", None)]:
            a = g.interior(name, stag)
            b = interior(o.f(name), nk, nj, ni, stag)
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (n, name)
    g.close()


@pytest.mark.parametrize("nk,kernel", [(40, "sound_slab"), (193, "sound_sub")])
def test_timer_names_the_kernel_that_runs(require_gpu, nk, kernel):
    import ctypes as C
    from cm1_amd import _native as N
    cfgd, cols, fields = case(ni=8, nj=8, nk=nk, dz=15000.0 / nk, dt=2.0, amp=2.0)
    g = make_gpu(cfgd, cols, fields)
    N.check(g.L.cm1g_ktimer_start(g.h, N.KT_SOUND_SUBSTEP), "cm1g_ktimer_start")
    g.step(1)
    ms, n, b, name = C.c_double(), C.c_int64(), C.c_double(), C.create_string_buffer(64)
    N.check(g.L.cm1g_ktimer_stop(g.h, C.byref(ms), C.byref(n), C.byref(b), name, 64), "cm1g_ktimer_stop")
    assert name.value.decode() == kernel and n.value == 2 + 3 + 6
    g.close()


BOX = ["u3d", "v3d", "w3d", "pp3d", "ppx", "rru", "rrv", "rrw"]


@pytest.mark.parametrize("we,sn", [(1, 1), (2, 2), (1, 2), (2, 1)], ids=["periodic", "open", "we-periodic", "sn-periodic"])
@pytest.mark.parametrize("ni,nj,nk,nsound", [(8, 9, 6, 2), (13, 8, 9, 5), (70, 11, 8, 10)])
def test_explicit_routine_whole_boxes(require_gpu, ni, nj, nk, nsound, we, sn):
    """sounde as a routine, every stage, from arrays that differ everywhere
    (borders too): whole boxes equal the oracle's."""
    import ctypes as C

    import pyoracle
    from cm1_amd import _native as N
    cfgd, cols, fields = case(ni=ni, nj=nj, nk=nk, nsound=nsound, dz=15000.0 / nk, dt=0.25 * nsound, amp=2.0, psolver=2)
    cfgd.update(wbc=we, ebc=we, sbc=sn, nbc=sn)
    g = make_gpu(cfgd, cols, fields)
    o = make_oracle(cfgd, cols, fields)
    g.step(1)  # (the open sides' radiation speeds)
    o.step(1)
    rng = np.random.default_rng(ni)
    noise = ("ua", "va", "wa", "ppi", "u3d", "v3d", "w3d", "pp3d", "ppx", "rru", "rrv", "rrw")
    for nrk in (1, 2, 3):
        for n in noise:
            o.f(n)[:] = (rng.standard_normal(o.f(n).shape) * 0.1).astype(np.float32)
        for n in pyoracle.FIELDS:
            g.put(n, np.ascontiguousarray(o.f(n)))
        dttmp = C.c_float(np.float32(cfgd["dt"]) / np.float32(4 - nrk))
        N.check(g.L.cm1g_sound(g.h, nrk, dttmp), "cm1g_sound")
        o.L.cm1o_sound(o.h, nrk, dttmp)
        for n in BOX:
            assert np.array_equal(g.get(n).view(np.uint32), o.f(n).view(np.uint32)), (nrk, n)
    g.close()


@pytest.mark.parametrize("we,sn", [(1, 1), (2, 2), (1, 2), (2, 1)], ids=["periodic", "open", "we-periodic", "sn-periodic"])
def test_explicit_step_whole_boxes(require_gpu, we, sn):
    """Whole steps with the explicit solver: what the halo fills leave in the
    corners comes from the border the substeps start from."""
    cfgd, cols, fields = case(ni=13, nj=9, nk=8, nsound=10, dz=15000.0 / 8, dt=2.0, amp=2.0, psolver=2)
    cfgd.update(wbc=we, ebc=we, sbc=sn, nbc=sn)
    g = make_gpu(cfgd, cols, fields)
    o = make_oracle(cfgd, cols, fields)
    for _ in range(3):  # from equal arrays, then from exchanged buffers
        g.step(1)
        o.step(1)
        for n in ("u3d", "v3d", "w3d", "pp3d"):
            assert np.array_equal(g.get(n).view(np.uint32), o.f(n).view(np.uint32)), n
    g.close()
