"""Start labels written by the device: sizes that leave a partial last word
group, given and own labels, seeds; label buffers and captured steps kept
from one run to the next; refused labels leave the state as it was."""
import numpy as np
import pytest

import lpa_amd as L
from gpu_common import run_and_compare

pytestmark = pytest.mark.gpu
UNL = 0xFFFFFFFF


def _engine(K, semi=False, scale=10, **cms):
    g = L.gen_copying(1003 if scale == 10 else 1 << scale, 12.0, 2.1, 500, 0.7, 50, seed=3)
    cgr = g.encode(0, 128)
    e = L.Engine(0)
    e.upload(cgr)
    e.config(K=K, semi=semi, **cms)
    e.schedule_degree()
    return g, cgr, e


@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 7, 8, 33])
@pytest.mark.parametrize("semi", [False, True])
def test_start_labels(K, semi):
    g, cgr, e = _engine(K, semi)
    e.labels_init()
    assert np.array_equal(e.labels(), np.repeat(np.arange(g.n, dtype=np.uint32), K))
    lab = np.random.default_rng(K).integers(0, 50, g.n * K).astype(np.uint32)
    lab[::3] = UNL
    e.labels_init(lab)
    assert np.array_equal(e.labels(), lab)
    run_and_compare(cgr, 3, labels0=lab, K=K, semi=semi, engine=e)
    # a run over the same buffers, one from own labels, and one with more vectors
    run_and_compare(cgr, 2, K=K, semi=semi, engine=e)
    e.config(K=K + 1, semi=semi)
    e.schedule_degree()
    run_and_compare(cgr, 2, K=K + 1, semi=semi, engine=e)
    e.close()


def test_captured_steps_survive_new_labels_but_not_new_parameters():
    cms = dict(cms_thresh=20, cms_depth=3, cms_width=64)
    g, cgr, e = _engine(2, cms_seed=1, **cms)
    e.set_graph_mode(True)
    for it in range(3):
        run_and_compare(cgr, 3, K=2, cms_seed=1, engine=e, **cms)
    lab = np.random.default_rng(1).integers(0, 9, g.n * 2).astype(np.uint32)
    run_and_compare(cgr, 3, labels0=lab, K=2, cms_seed=1, engine=e, **cms)
    # other row hashes, same layout
    e.config(K=2, cms_seed=7, **cms)
    run_and_compare(cgr, 4, labels0=lab, K=2, cms_seed=7, engine=e, **cms)
    e.close()


def test_refused_labels_leave_the_state():
    g, cgr, e = _engine(2)
    e.labels_init()
    e.nova_iterate()
    before = e.labels()
    bad = np.zeros(g.n * 2, np.uint32)
    bad[-1] = 0x80000000
    with pytest.raises(L.LpaError):
        e.labels_init(bad)
    assert np.array_equal(e.labels(), before)
    e.nova_iterate()
    run_and_compare(cgr, 2, K=2, engine=e)
    e.close()
