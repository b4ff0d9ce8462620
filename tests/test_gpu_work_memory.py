"""Working memory too large to keep goes back when a call ends, also when the
call is refused."""
import numpy as np
import pytest
import torch

import lpa_amd as L

pytestmark = pytest.mark.gpu


def test_refused_encode_gives_its_memory_back():
    n, d = 1 << 20, 67
    row = np.arange(n + 1, dtype=np.uint64) * d
    col = np.tile(np.arange(d, dtype=np.uint32) * 15000, n)
    col[-2:] = col[-2:][::-1].copy()      # the last row is out of order
    assert col.nbytes > 256 << 20         # more than an engine keeps of one buffer
    e = L.Engine(0)
    g = L.gen_rmat(10, 8, seed=1)
    e.encode_csr(g.row, g.col, 0)
    before = torch.cuda.mem_get_info(0)[0]
    with pytest.raises(L.LpaError, match="strictly increasing"):
        e.encode_csr(row, col, 0)
    assert before - torch.cuda.mem_get_info(0)[0] < 128 << 20
    e.encode_csr(g.row, g.col, 0)         # and the engine goes on
    assert e.stream()[3] == g.encode(0, 128).nbits
