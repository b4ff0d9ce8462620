"""One heavy set with one-workgroup and chunked vertices: the hubs' chunks run
on the second side stream, behind the decode of their lists, beside the
one-workgroup vertices on the first; eager, and forked inside a captured step."""
import numpy as np
import pytest

import lpa_amd as L
from gpu_common import make_engine, run_and_compare

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hubs():
    n, rng = 40_000, np.random.default_rng(5)
    src, dst = [rng.integers(0, n, 6 * n)], [rng.integers(0, n, 6 * n)]
    for v, d in ((17, 30_000), (901, 12_000), (2222, 9_000), (5, 7_000), (30_000, 6_000), (39_999, 3_000)):
        src.append(np.full(d, v))
        dst.append(rng.choice(n, d, replace=False))
    src, dst = np.concatenate(src).astype(np.uint32), np.concatenate(dst).astype(np.uint32)
    g = L.Csr.from_edges(n, np.concatenate([src, dst]), np.concatenate([dst, src]), False)
    d = g.degrees()
    # exact hubs of one workgroup (above 2048 ids) and of several (above 8192)
    assert ((d > 2048) & (d <= 8192)).sum() >= 3 and (d > 8192).sum() >= 3
    return g


@pytest.mark.parametrize("method", ["nova", "cglp", "csr"])
@pytest.mark.parametrize("K", [1, 8])
def test_eager(hubs, method, K):
    cgr = hubs.encode(0, 128)
    e = make_engine(cgr, K=K)
    assert e.counts()["global"] >= 6 and not e.counts()["cms"]
    for _ in range(2):
        run_and_compare(cgr, 4, method=method, K=K, engine=e)


@pytest.mark.parametrize("K", [8, 17])
def test_captured(hubs, K):
    cgr = hubs.encode(0, 128)
    e = make_engine(cgr, K=K)
    assert hubs.m * K > 4 << 20   # label reads from which a captured step forks
    for rep in range(3):
        e.set_graph_mode(True)
        run_and_compare(cgr, 4, K=K, engine=e)
        run_and_compare(cgr, 3, method="cglp", K=K, engine=e)
        if rep == 1:
            e.set_graph_mode(False)
            run_and_compare(cgr, 2, K=K, engine=e)
