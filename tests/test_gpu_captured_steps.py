"""Captured steps whose buffers move between two uses: the stream goes to
host memory and back while captured steps of it exist."""
import pytest

import lpa_amd as L
from gpu_common import make_engine, run_and_compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,method", [(1, "nova"), (8, "nova"), (2, "cglp")])
def test_stream_moved_after_a_timed_capture(K, method):
    g = L.gen_rmat(13, 16, seed=11)
    cgr = g.encode(0, 128)
    e = make_engine(cgr, K=K)
    e.labels_init()
    e.time_iterations(2, method, use_graph=True)   # graph mode itself stays off
    e.stream_residence(True, 1 << 16)
    keep = L.Engine(0)                              # takes what the stream gave back
    keep.upload(L.gen_rmat(13, 16, seed=12).encode(0, 128))
    e.stream_residence(False)
    e.set_graph_mode(True)
    run_and_compare(cgr, 4, K=K, method=method, engine=e)
    # and with eager steps in between
    e.set_graph_mode(False)
    run_and_compare(cgr, 2, K=K, method=method, engine=e)
