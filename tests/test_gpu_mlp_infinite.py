"""Gradients where activations or weights are not finite: a factor of 0 (an
output that was not measured, a unit that is off) takes no part, whatever it
would be multiplied by."""
import numpy as np
import pytest

import lpa_amd as L
import mlp_ref as R
from test_gpu_mlp_order import F, _fma, _walk

pytestmark = pytest.mark.gpu


def _back(w, d):
    z = np.zeros((len(d), w.shape[1]), F)
    for j in range(w.shape[0]):
        z = np.where(d[:, j:j + 1] == 0, z, _fma(d[:, j:j + 1], w[j], z))
    return z


def _grad(p, x, t, mask):
    w = {k: v.astype(F) for k, v in R.unpack(p).items()}
    z1 = _walk(w["W1"], w["b1"], x)
    h1 = np.where(z1 > 0, z1, F(0))
    z2 = _walk(w["W2"], w["b2"], h1)
    h2 = np.where(z2 > 0, z2, F(0))
    dy = F(2) * np.where(mask, _walk(w["W3"], w["b3"], h2) - t, F(0)) * (F(1) / F(len(x)))
    d2 = np.where(h2 > 0, _back(w["W3"], dy), F(0))
    d1 = np.where(h1 > 0, _back(w["W2"], d2), F(0))

    def outer(d, v):
        return np.where(d[:, :, None] == 0, F(0), d[:, :, None] * v[:, None]).reshape(len(x), -1)

    g = np.zeros(R.NPARAM, F)
    for term in np.concatenate([outer(d1, x), d1, outer(d2, h1), d2, outer(dy, h2), dy], 1):
        g += term
    return g


@pytest.mark.parametrize("case", ["inputs", "activations", "third layer", "second layer"])
def test_factors_of_zero(case):
    rng = np.random.default_rng(4)
    n = 50
    p = rng.normal(0, 0.3, R.NPARAM).astype(F)
    x, t = rng.normal(0, 1, (n, 8)).astype(F), rng.normal(0, 1, (n, 3)).astype(F)
    mask = rng.random((n, 3)) < 0.7
    mask[7] = [True, False, False]
    if case == "inputs":
        x[7, 3] = np.inf
    elif case == "activations":
        x[7] *= F(3e38) / np.abs(x[7]).max()
    elif case == "third layer":   # an output that is measured nowhere
        p[1344 + 32:1344 + 64] = np.inf
        mask[:, 1] = False
    else:                         # a unit that is always off
        p[288 + 5 * 32:288 + 6 * 32] = -np.inf
    m = L.Mlp(0, seed=3)
    m.params = p
    with np.errstate(all="ignore"):
        want = _grad(p, x, t, mask)
    assert np.isfinite(want).sum() >= 67   # at least two outputs' weights and biases
    assert np.array_equal(m.loss_grad(x, t, mask)[1], want, equal_nan=True)
