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
