"""Heavy sets on side streams: eager steps (all three methods), captured steps
large enough to fork inside the graph, replayed several times with eager steps
between, and the change counts of all streams."""
import pytest

import lpa_amd as L
from gpu_common import make_engine, run_and_compare

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rmat15():
    return L.gen_rmat(15, 20, seed=9).encode(16, 128)


# degrees 2049..4096 count exactly, above with sketches: two heavy sets
CMS = dict(cms_thresh=4096, cms_depth=3, cms_width=512, cms_seed=2)


@pytest.mark.parametrize("method", ["nova", "cglp", "csr"])
@pytest.mark.parametrize("K", [1, 3])
def test_eager(rmat15, method, K):
    e = make_engine(rmat15, K=K, **CMS)
    c = e.counts()
    assert c["global"] and c["cms"]
    for _ in range(2):
        run_and_compare(rmat15, 4, method=method, K=K, engine=e, **CMS)
    # another method on the same engine, and timed steps on one stream between
    e.time_iterations(2, method)
    run_and_compare(rmat15, 2, method="nova", K=K, engine=e, **CMS)
    e.close()


@pytest.mark.parametrize("K,cms", [(8, CMS), (8, {}), (17, CMS)])
def test_captured(rmat15, K, cms):
    e = make_engine(rmat15, K=K, **cms)
    assert rmat15.nbits and K * 1_000_000 > 4 << 20   # about 1.1 M arcs: the graph forks
    for rep in range(3):
        e.set_graph_mode(True)
        run_and_compare(rmat15, 5, K=K, engine=e, **cms)
        run_and_compare(rmat15, 3, method="cglp", K=K, engine=e, **cms)
        if rep == 1:
            e.set_graph_mode(False)
            run_and_compare(rmat15, 2, K=K, engine=e, **cms)
    e.close()
