"""Timed steps are the steps that the iterate entry points run: the same
labels and change counts, and about the same time."""
import time

import numpy as np
import pytest

import lpa_amd as L
import pyoracle as O
from gpu_common import make_engine, oracle_view

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method", ["nova", "cglp", "csr"])
@pytest.mark.parametrize("K,use_graph", [(1, False), (8, False), (3, True)])
def test_labels_and_counts_of_timed_steps(method, K, use_graph):
    g = L.gen_rmat(13, 16, seed=11)
    cgr = g.encode(0, 128)
    e = make_engine(cgr, K=K, cms_thresh=512)
    e.labels_init()
    ms, changed = e.time_iterations(4, method, use_graph=use_graph)
    view, c = oracle_view(cgr), O.cfg(K=K, cms_thresh=512, cms_depth=4, cms_width=1024, cms_seed=0)
    lab = np.repeat(np.arange(cgr.n, dtype=np.uint32), K)
    for it in range(4):
        lab, och = O.step_cgr(view, lab, c)
        assert changed[it] == och and ms[it] > 0
    assert np.array_equal(e.labels(), lab)
    if method == "nova" and not use_graph:
        kt = e.kernel_times()
        assert all(kt[k] > 0 for k, s in e.stats().items() if s["vertices"] and k != "skip")
    # and the step after them
    e.nova_iterate()
    lab, _ = O.step_cgr(view, lab, c)
    assert np.array_equal(e.labels(), lab)


def test_timed_step_is_the_step_that_runs():
    """a small graph, whose step is a few launches where every bin by itself
    makes a dozen: the fastest of 40 on either clock, the device's timestamps
    within half of the host's time"""
    e = make_engine(L.gen_rmat(12, 16, seed=1).encode(0, 128), K=1, cms_thresh=256, cms_width=512)
    e.labels_init()
    for _ in range(5):
        e.nova_iterate()
    host = []
    for _ in range(40):
        t = time.perf_counter()
        e.nova_iterate()
        host.append((time.perf_counter() - t) * 1e3)
    ms, _ = e.time_iterations(40)
    assert ms.min() <= 1.5 * min(host), (ms.min(), min(host))
