"""Columns cut into segments by the marching kernels (advection, mass fluxes,
the positive-definite pass): level counts around the segment lengths, where
the one-sided boundary fluxes meet a segment's first and last level, against
the oracle bit for bit."""
import numpy as np
import pytest

from common import PROG, case, interior, make_gpu, make_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("opts", [
    dict(bc=2, npt=1),
    dict(bc=2, advwenos=1, advwenov=1, npt=1),
    dict(bc=1, psolver=2, nsound=10, advwenos=2, advwenov=2),
], ids=["flx5", "weno", "weno-last"])
@pytest.mark.parametrize("nk", [6, 7, 8, 9, 12, 13, 17, 23, 31, 50])
def test_segment_edges_match_oracle(require_gpu, nk, opts):
    ni, nj = 13, 9
    cfgd, cols, fields = case(ni=ni, nj=nj, nk=nk, dz=15000.0 / nk, dt=4.0, amp=2.0, seed=nk, **opts)
    if opts.get("npt"):
        rng = np.random.default_rng(nk)
        fields["pta0"][1:nk + 1, 3:nj + 3, 3:ni + 3] = rng.uniform(0.0, 1.0, (nk, nj, ni)).astype(np.float32)
    g = make_gpu(cfgd, cols, fields)
    o = make_oracle(cfgd, cols, fields)
    g.step(2)
    o.step(2)
    for name, stag in PROG + [(f"pta{t}", None) for t in range(opts.get("npt", 0))]:
        a = g.interior(name, stag)
        b = interior(o.f(name), nk, nj, ni, stag)
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), name
    g.close()
