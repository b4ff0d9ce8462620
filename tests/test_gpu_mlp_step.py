"""The cost model's training step on the matrix cores against the float64
reference: sample counts around the 16-sample tiles, the 64-sample workgroups
and the limits on the number of workgroups, samples without a measured output,
and several Adam steps with a ragged last batch."""
import numpy as np
import pytest

import lpa_amd as L
import mlp_ref as R

pytestmark = pytest.mark.gpu

MASK64 = (1 << 64) - 1


def _data(n, seed):
    rng = np.random.default_rng(seed)
    p = rng.normal(0, 0.25, R.NPARAM).astype(np.float32)
    x = rng.normal(0, 1, (n, 8)).astype(np.float32)
    t = rng.normal(0, 1, (n, 3)).astype(np.float32)
    mask = rng.random((n, 3)) < 0.7
    mask[0] = True
    return p, x, t, mask


# 64 samples per workgroup, at most 256 workgroups: 16384 + 1 wraps
@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 129, 16384, 16385])
def test_gradient_sizes(n):
    p, x, t, mask = _data(n, n)
    m = L.Mlp(0, seed=1)
    m.params = p
    loss, g = m.loss_grad(x, t, mask)
    want_l, want_g = R.loss_grad(p.astype(np.float64), x.astype(np.float64), t.astype(np.float64), mask)
    assert abs(loss - want_l) <= 1e-5 * abs(want_l)
    # float32 sums: relative to the largest element of the gradient
    assert np.abs(g - want_g).max() <= 1e-5 * np.abs(want_g).max()


def test_unmeasured_samples_may_hold_anything():
    """a sample whose outputs are all masked out contributes nothing, even
    when its features are not finite"""
    p, x, t, mask = _data(100, 5)
    mask[[3, 50, 99]] = False
    m = L.Mlp(0, seed=1)
    m.params = p
    want = m.loss_grad(x, t, mask)
    x[3], x[50, 2], x[99, 7] = np.nan, np.inf, -np.inf
    t[3] = np.nan
    got = m.loss_grad(x, t, mask)
    assert got[0] == want[0] and np.array_equal(got[1], want[1])


def _shuffled(idx, s):
    idx = idx.copy()
    for i in range(len(idx) - 1, 0, -1):
        s = (s + 0x9E3779B97F4A7C15) & MASK64
        z = ((s ^ (s >> 30)) * 0xBF58476D1CE4E5B9) & MASK64
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & MASK64
        z ^= z >> 31
        j = z % (i + 1)
        idx[i], idx[j] = idx[j], idx[i]
    return idx, s


# one workgroup; several with a ragged last batch; more samples than the 64
# workgroups of a training step take at once (4096)
@pytest.mark.parametrize("n,batch,epochs", [(70, 32, 2), (1000, 300, 2), (9000, 4500, 1)])
def test_adam_steps(n, batch, epochs):
    p, x, t, mask = _data(n, 7)
    m = L.Mlp(0, seed=1)
    m.params = p
    lr, seed = 1e-3, 11
    losses = m.train(x, t, mask, epochs=epochs, batch=batch, lr=lr, seed=seed)
    q = p.astype(np.float64)
    m1, m2, k = np.zeros(R.NPARAM), np.zeros(R.NPARAM), 0
    idx, s, want = np.arange(n), seed, []
    small = np.zeros(R.NPARAM, bool)   # elements whose gradient drowns in rounding at some step
    for _ in range(epochs):
        idx, s = _shuffled(idx, s)
        ls = []
        for b0 in range(0, n, batch):
            b = idx[b0:b0 + batch]
            l, g = R.loss_grad(q, x[b].astype(np.float64), t[b].astype(np.float64), mask[b])
            ls.append(l)
            small |= np.abs(g) < 1e-3 * np.abs(g).max()
            k += 1
            m1, m2 = 0.9 * m1 + 0.1 * g, 0.999 * m2 + 0.001 * g * g
            q = q - lr * (m1 / (1 - 0.9 ** k)) / (np.sqrt(m2 / (1 - 0.999 ** k)) + 1e-8)
        want.append(np.mean(ls))
    assert np.allclose(losses, want, rtol=1e-4)
    d = np.abs(m.params - q)
    # an Adam step moves a parameter by about lr; its relative error is that
    # of the gradient element (1e-5 of the largest element, so at most 1 % of
    # those above 1e-3 of it)
    assert (d[~small] <= 1e-2 * lr * k + 1e-6).all(), d[~small].max()
    assert (d <= 2 * lr * k + 1e-6).all()
