"""Half-wave groups over lists of 129 to 512 ids (quarter_max above its
default), beside bins that need less LDS, against the oracle."""
import pytest

import lpa_amd as L
from gpu_common import run_and_compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [3, 5, 8, 9])
@pytest.mark.parametrize("quarter_max", [256, 300])
def test_wide_half_waves(K, quarter_max):
    g = L.gen_rmat(13, 16, seed=11)
    d = g.degrees()
    assert ((d > 128) & (d <= 256)).sum() > 100
    run_and_compare(g.encode(0, 128), 3, K=K, lane_max=8, quarter_max=quarter_max)
