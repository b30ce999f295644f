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


def test_silu_derivative_in_single_precision(require_gpu):
    """One row through a network whose third layer sees its biases alone (all
    hidden weights 0) and whose output weights and output error make that
    layer's bias gradient SiLU's derivative at those biases, unrounded.

    Tolerance, with u = 2^-24: exp within an ulp (2u), the sum and the division
    rounded (u each), so the sigmoid s is within 4u of itself; q = 1 + z(1 - s)
    takes in 4us|z| from s and 2u|z| from two roundings, and rounds itself (u
    |q|), as the product s q does."""
    import torch
    z = np.linspace(-80.0, 20.0, R.NH).astype(np.float32)
    z[-1] = 0.0
    net = S.Net(seed=1)
    w = {name: np.zeros(shape) for name, shape in R.SIZES}
    w["b3"] = z
    w["W4"][:, 0] = 1.0
    net.set_params(R.pack(w))
    x = torch.ones((1, 8), device="cuda")
    t = net.forward(x)
    t[0, 0] -= 2.0  # 2 (y - t) / 4 = 1
    _, g = net.loss_grad(x, t, want_grad=True)
    at = sum(int(np.prod(s)) for _, s in R.SIZES[:5])
    d = g[at:at + R.NH].astype(np.float64)
    net.close()
    z = z.astype(np.float64)
    s = 1.0 / (1.0 + np.exp(-z))
    # (z < 0: 1 - s without its cancellation)
    q = 1.0 + z / (1.0 + np.exp(z))
    u = 2.0 ** -24
    tol = s * (4 * u * np.abs(q) + np.abs(z) * (4 * u * s + 2 * u) + 2 * u * np.abs(q)) + 2.0 ** -149
    assert d[-1] == 0.5
    assert (np.abs(d - s * q) <= tol).all(), np.max(np.abs(d - s * q) / tol)


def test_loss_adds_up_over_many_groups(require_gpu):
    """All weights 0: every squared error is that of the target, whose sum over
    a wavefront's many groups would drift in single precision.  Tolerance: a
    square, three sums of a sample's four and the result rounded to single."""
    import torch
    rows, c = 2 ** 21 + 3, np.float32(0.7325)
    drift = np.cumsum(np.full(256, c * c, np.float32), dtype=np.float32)[-1] / (256 * float(c) ** 2) - 1.0
    assert abs(drift) > 1.0e-6
    net = S.Net(seed=2)
    net.set_params(np.zeros(R.NPARAM, np.float32))
    x = torch.ones((rows, 8), device="cuda")
    t = torch.full((rows, 4), float(c), device="cuda")
    loss = net.loss_grad(x, t)
    net.close()
    assert abs(loss / float(c) ** 2 - 1.0) <= 5 * 2.0 ** -24


def test_many_groups_a_wavefront(require_gpu):
    """Eight 16-sample groups for most wavefronts, a last one that is not full."""
    import torch
    rows = 2 ** 18 + 5
    rng = np.random.default_rng(rows)
    net = S.Net(seed=3)
    x = rng.standard_normal((rows, 8)).astype(np.float32)
    t = rng.standard_normal((rows, 4)).astype(np.float32)
    loss, g = net.loss_grad(torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda(), want_grad=True)
    loss_r, g_r = R.loss_grad(net.params().astype(np.float64), x.astype(np.float64), t.astype(np.float64), rnd=True)
    net.close()
    assert abs(loss - loss_r) <= TOL * loss_r, (loss, loss_r)
    offs = np.cumsum([0] + [int(np.prod(s)) for _, s in R.SIZES])
    for (name, _), a, b in zip(R.SIZES, offs[:-1], offs[1:]):
        assert rel(g[a:b], g_r[a:b]) < TOL, name
