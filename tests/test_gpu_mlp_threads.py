"""One model used by several threads at once: predictions (through the
runtime's copies and through the pinned slots) and gradients, each thread's
results those of its own inputs."""
import threading

import numpy as np
import pytest

import lpa_amd as L
import mlp_ref as R

pytestmark = pytest.mark.gpu


def test_threads_share_a_model():
    rng = np.random.default_rng(1)
    m = L.Mlp(0, seed=1)
    m.params = rng.normal(0, 0.3, R.NPARAM).astype(np.float32)
    sizes = [1000, 30_001, 300_000, 400_007]
    xs = [rng.normal(0, 1, (n, 8)).astype(np.float32) for n in sizes]
    t = rng.normal(0, 1, (5000, 3)).astype(np.float32)
    mask = np.ones((5000, 3), bool)
    m.forward(np.zeros((1 << 21, 8), np.float32))   # 64 MB: the slots are in use from here on
    want = [m.forward(x) for x in xs]
    want_g = m.loss_grad(xs[1][:5000], t, mask)
    bad = []

    def predict(i):
        for _ in range(12):
            if not np.array_equal(m.forward(xs[i]), want[i]):
                bad.append(sizes[i])

    def gradient():
        for _ in range(30):
            loss, g = m.loss_grad(xs[1][:5000], t, mask)
            if loss != want_g[0] or not np.array_equal(g, want_g[1]):
                bad.append("gradient")

    threads = [threading.Thread(target=predict, args=(i,)) for i in range(len(xs))] + [threading.Thread(target=gradient)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not bad
