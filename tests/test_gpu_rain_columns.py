"""The Kessler branch's column work (rescaling of clipped water, fall speeds,
sedimentation) holds 64 columns of a row in LDS: level counts around what its
wavefronts and its LDS sizes hold, deeper columns, ragged rows and several
sedimentation substeps, against the oracle bit for bit."""
import numpy as np
import pytest

from cm1_amd import _native as N
from common import case, make_gpu, make_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nk", [6, 15, 16, 17, 48, 49, 64, 65, 96, 97, 128, 129])
def test_rain_columns(require_gpu, nk):
    ni, nj = (65, 8) if nk % 2 else (9, 10)
    cfgd, cols, fields = case(ni=ni, nj=nj, nk=nk, dz=20.0, dt=6.0)
    g = make_gpu(cfgd, cols, fields)
    o = make_oracle(cfgd, cols, fields)
    rng = np.random.default_rng(nk)
    for n, hi in (("q3d0", 1.0e-2), ("q3d1", 1.0e-3), ("q3d2", 1.0e-2)):
        a = rng.uniform(0.0, hi, (o.pz, o.py, o.px)).astype(np.float32)
        kind = rng.integers(0, 12, a.shape)
        a[kind == 0] = -1.0e-5
        a[kind == 1] = -0.0
        a[kind == 2] = 0.0
        a[kind == 3] = 1.0e-9
        a[:, 3] = np.abs(a[:, 3]) + np.float32(1.0e-6)  # a row with nothing to clip
        o.f(n)[:] = a
        g.put(n, a)
    for n in ("rho", "th3d", "pp3d", "prs"):
        g.put(n, np.ascontiguousarray(o.f(n)))
    N.check(g.L.cm1g_kessler_branch(g.h), "cm1g_kessler_branch")
    o.L.cm1o_kessler_branch(o.h)
    for n in ("q3d0", "q3d1", "q3d2", "th3d", "pp3d", "prs"):
        a, b = g.get(n), o.f(n)
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), n
    # (the domain budget adds a column's substeps up before the columns, the
    # oracle goes on through the row; with one substep a column they are the
    # same sum, test_kessler_branch_signed_zeros)
    for n in ("rain", "prate"):
        a = np.empty((nj + 6, ni + 6), np.float32)
        N.check(g.L.cm1g_get_2d_array(g.h, N.D2[n], a.ctypes.data), "cm1g_get_2d_array")
        a, b = (np.ascontiguousarray(x[3:nj + 3, 3:ni + 3]) for x in (a, o.d2(n)))
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)) and a.any(), n
    g.close()
