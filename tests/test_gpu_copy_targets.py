"""Large copies to and from memory that is not ordinary pages, once copies go
through the pinned slots: the stream into device memory and into pinned
memory, predictions between pinned arrays."""
import ctypes as C

import numpy as np
import pytest
import torch

import lpa_amd as L
import mlp_ref as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("host_resident", [False, True])
def test_stream_into_device_and_pinned_memory(host_resident):
    g = L.gen_rmat(18, 16, seed=3)
    e = L.Engine(0)
    if host_resident:
        e.stream_residence(True)
    e.upload(g.encode(0, 128))
    words = e.stream()[0]
    assert words.nbytes > 8 << 20
    for _ in range(8):   # 64 MB: the slots are in use from here on
        assert np.array_equal(e.stream()[0], words)
    n_c, nbits = C.c_uint64(), C.c_uint64()
    for t in (torch.zeros(len(words), dtype=torch.int64, device="cuda:0"),
              torch.zeros(len(words), dtype=torch.int64, pin_memory=True)):
        torch.cuda.synchronize()
        rc = e._L.lpa_graph_stream(e._h, C.byref(n_c), C.byref(nbits), C.c_void_p(t.data_ptr()), None, None)
        assert rc == 0
        assert np.array_equal(t.cpu().numpy().view(np.uint64), words)


def test_predictions_between_pinned_arrays():
    rng = np.random.default_rng(2)
    m = L.Mlp(0, seed=1)
    m.params = rng.normal(0, 0.3, R.NPARAM).astype(np.float32)
    n = 1 << 19
    x = rng.normal(0, 1, (n, 8)).astype(np.float32)
    for _ in range(5):
        want = m.forward(x)
    px = torch.from_numpy(x).pin_memory()
    py = torch.zeros((n, 3), dtype=torch.float32, pin_memory=True)
    rc = m._L.lpa_mlp_forward(m._h, C.c_void_p(px.data_ptr()), n, C.c_void_p(py.data_ptr()))
    assert rc == 0 and np.array_equal(py.numpy(), want)
