"""The surrogate's gradients and inference at row counts around its 16-sample
groups, pairs of groups and workgroups, and from rows that start on any float,
against the CPU oracle of the network.

Tolerance: both sides round the operands of every product to BF16 (8 bits of
mantissa), so a value that lies on a rounding boundary may fall either way:
no operand is off by more than 2^-8 of itself.
"""
import numpy as np
import pytest

import mlp_ref as R
from cm1_amd import surrogate as S

pytestmark = pytest.mark.gpu
TOL = 2.0 ** -8


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(b))


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 33, 127, 129, 2049, 33000])
def test_gradients_and_forward(require_gpu, rows):
    import torch
    rng = np.random.default_rng(rows)
    net = S.Net(seed=rows)
    flat = rng.standard_normal(rows * 12 + 2).astype(np.float32)
    x, t = flat[1:1 + 8 * rows].reshape(rows, 8), flat[2 + 8 * rows:].reshape(rows, 4)
    dev = torch.from_numpy(flat).cuda()
    xd, td = dev[1:1 + 8 * rows].view(rows, 8), dev[2 + 8 * rows:].view(rows, 4)
    for step in range(2):  # with the first parameters, and after an Adam step
        p = net.params().astype(np.float64)
        loss, g = net.loss_grad(xd, td, want_grad=True)
        loss_r, g_r = R.loss_grad(p, x.astype(np.float64), t.astype(np.float64), rnd=True)
        assert abs(loss - loss_r) <= TOL * loss_r, (loss, loss_r)
        offs = np.cumsum([0] + [int(np.prod(s)) for _, s in R.SIZES])
        for (name, _), a, b in zip(R.SIZES, offs[:-1], offs[1:]):
            assert rel(g[a:b], g_r[a:b]) < TOL, (step, name)
        y = net.forward(xd).cpu().numpy()
        assert rel(y, R.forward(p, x.astype(np.float64), rnd=True)[0]) < TOL
        net.train(xd, td, steps=1, batch=rows)
    net.close()
