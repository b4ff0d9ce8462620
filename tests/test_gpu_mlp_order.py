"""The training step takes every sum in the order of a lane that walks over
the layers sample by sample, bit for bit: where a unit's pre-activation is a
rounding away from 0, another order switches the unit on or off, and training
ends elsewhere."""
import numpy as np
import pytest

import lpa_amd as L
import mlp_ref as R
from test_gpu_mlp_step import _shuffled

pytestmark = pytest.mark.gpu

F = np.float32


@pytest.mark.parametrize("n", [1, 16, 100, 5000])
def test_outputs_as_targets_leave_no_error(n):
    rng = np.random.default_rng(n)
    m = L.Mlp(0, seed=3)
    m.params = rng.normal(0, 0.4, R.NPARAM).astype(F)
    x = (rng.normal(0, 1, (n, 8)) * 10.0 ** rng.integers(-3, 3, (n, 8))).astype(F)
    loss, g = m.loss_grad(x, m.forward(x), np.ones((n, 3), bool))
    assert loss == 0 and not g.any()


def _fma(a, b, c):
    """float32 fused multiply-add (the product of two is exact in 64 bits)"""
    return (np.asarray(a, np.float64) * b + c).astype(F)


def _walk(w, b, x):
    """b + w x, inputs in ascending order; x: a row per sample"""
    z = np.broadcast_to(b, (len(x), len(b)))
    for i in range(w.shape[1]):
        z = _fma(x[:, i:i + 1], w[:, i], z)
    return z


def _grad(p, x, t, mask):
    w = {k: v.astype(F) for k, v in R.unpack(p).items()}
    z1 = _walk(w["W1"], w["b1"], x)
    h1 = np.maximum(z1, 0)
    z2 = _walk(w["W2"], w["b2"], h1)
    h2 = np.maximum(z2, 0)
    e = np.where(mask, _walk(w["W3"], w["b3"], h2) - t, F(0))
    dy = F(2) * e * (F(1) / F(len(x)))
    zero = np.zeros(32, F)
    d2 = np.where(h2 > 0, _walk(w["W3"].T, zero, dy), F(0))
    d1 = np.where(h1 > 0, _walk(w["W2"].T, zero, d2), F(0))
    terms = np.concatenate([(d1[:, :, None] * x[:, None]).reshape(len(x), -1), d1,
                            (d2[:, :, None] * h1[:, None]).reshape(len(x), -1), d2,
                            (dy[:, :, None] * h2[:, None]).reshape(len(x), -1), dy], 1)
    # 64 samples one after the other, four such sums, then those
    g = np.zeros(R.NPARAM, F)
    for b in range(0, len(x), 256):
        s = np.zeros(R.NPARAM, F)
        for c in range(b, min(b + 256, len(x)), 64):
            q = np.zeros(R.NPARAM, F)
            for term in terms[c:c + 64]:
                q += term
            s += q
        g += s
    return g, z1, z2


@pytest.mark.parametrize("seed", range(4))
def test_units_a_rounding_away_from_zero(seed):
    """samples that are all alike, and whose units all have a pre-activation
    of rounding size"""
    rng = np.random.default_rng(seed)
    w = {k: rng.normal(0, 0.5, s).astype(F) for k, s in R.SIZES}
    x = np.repeat(rng.normal(0, 4, (1, 8)).astype(F), 5, 0)
    w["b1"] = -(x[0].astype(np.float64) @ w["W1"].T).astype(F)
    w["b1"][::2] += F(0.5)   # half the first layer's units are on, so that the second has inputs
    h1 = np.maximum(_walk(w["W1"], w["b1"], x[:1]), 0)
    w["b2"] = -(h1[0].astype(np.float64) @ w["W2"].T).astype(F)
    p = np.concatenate([w[k].ravel() for k, _ in R.SIZES])
    t = rng.normal(0, 1, (5, 3)).astype(F)
    mask = np.ones((5, 3), bool)
    want, z1, z2 = _grad(p, x, t, mask)
    assert (np.abs(z1[:, 1::2]) < 1e-5).all() and (np.abs(z2) < 1e-5).all()
    assert (z2 > 0).any() and (z2 <= 0).any() and (z1[:, 1::2] <= 0).any()
    m = L.Mlp(0, seed=3)
    m.params = p
    assert np.array_equal(m.loss_grad(x, t, mask)[1], want)


# a part of a workgroup's 64 samples, several, and more than four of them
@pytest.mark.parametrize("n", [17, 64, 150, 600])
def test_gradient_bits(n):
    rng = np.random.default_rng(n)
    p = rng.normal(0, 0.3, R.NPARAM).astype(F)
    x, t = rng.normal(0, 1, (n, 8)).astype(F), rng.normal(0, 1, (n, 3)).astype(F)
    mask = rng.random((n, 3)) < 0.7
    m = L.Mlp(0, seed=3)
    m.params = p
    assert np.array_equal(m.loss_grad(x, t, mask)[1], _grad(p, x, t, mask)[0])


@pytest.mark.parametrize("n,batch,epochs", [(40, 40, 3), (500, 300, 2)])
def test_parameter_bits(n, batch, epochs):
    rng = np.random.default_rng(n)
    p = rng.normal(0, 0.3, R.NPARAM).astype(F)
    x, t = rng.normal(0, 1, (n, 8)).astype(F), rng.normal(0, 1, (n, 3)).astype(F)
    mask = rng.random((n, 3)) < 0.7
    m = L.Mlp(0, seed=3)
    m.params = p
    m.train(x, t, mask, epochs=epochs, batch=batch, lr=2e-3, seed=5)
    b1, b2, lr, eps = F(0.9), F(0.999), F(2e-3), F(1e-8)
    m1, m2, k, idx, s = np.zeros(R.NPARAM, F), np.zeros(R.NPARAM, F), 0, np.arange(n), 5
    for _ in range(epochs):
        idx, s = _shuffled(idx, s)
        for b0 in range(0, n, batch):
            b = idx[b0:b0 + batch]
            g = _grad(p, x[b], t[b], mask[b])[0]
            k += 1
            m1 = _fma(F(1) - b1, g, b1 * m1)
            m2 = _fma(g, (F(1) - b2) * g, b2 * m2)
            c1, c2 = F(1 / (1 - float(b1) ** k)), F(1 / (1 - float(b2) ** k))
            p = p - lr * (m1 * c1) / (np.sqrt(m2 * c2) + eps)
    assert np.array_equal(m.params, p)
