"""Large copies between host memory and the device (several threads from 64 MB
on): sizes around the 2 MiB chunks and the limits, first and repeated calls,
and working memory that grows and shrinks from call to call."""
import numpy as np
import pytest

import lpa_amd as L
import mlp_ref as R

pytestmark = pytest.mark.gpu


def _model():
    m = L.Mlp(0, seed=2)
    rng = np.random.default_rng(0)
    p = rng.normal(0, 0.2, R.NPARAM).astype(np.float32)
    m.params = p
    return m, p


def test_forward_sizes():
    # 32 bytes in and 12 out per sample: 8 MiB in is 262,144 samples, a chunk
    # out 174,763; the same model goes through all of them, large and small
    m, p = _model()
    rng = np.random.default_rng(1)
    big = rng.normal(0, 1, (2_200_000, 8)).astype(np.float32)
    want = R.forward(p.astype(np.float64), big.astype(np.float64))[0]
    bound = 1e-5 * (1 + np.abs(want).max())
    for n in (2_200_000, 10, 262_143, 262_144, 262_145, 349_525, 349_526, 1_048_577, 2_200_000, 1):
        y = m.forward(big[:n])
        assert y.shape == (n, 3) and np.abs(y - want[:n]).max() <= bound, n
        # other inputs in the same memory
        y2 = m.forward(big[:n][::-1])
        assert np.array_equal(y2[::-1], y), n


@pytest.mark.parametrize("semi", [False, True])
def test_labels_round_trip(semi):
    """labels in and out, 80 MB and a ragged size, and small ones after them"""
    rng = np.random.default_rng(3)
    for n, K in ((1_250_003, 16), (1_250_003, 3), (1_250_003, 1)):
        row = np.zeros(n + 1, np.uint64)
        row[2:] = 1                                # one arc: 1 -> 0
        e = L.Engine(0)
        e.upload(L.Csr.from_arrays(row, np.zeros(1, np.uint32)).encode(0, 128))
        e.config(K=K, semi=semi)
        e.schedule_degree()
        for _ in range(2):
            lab = rng.integers(0, 1 << 31, n * K, dtype=np.uint32)
            lab[rng.random(n * K) < 0.3] = 0xFFFFFFFF
            e.labels_init(lab)
            assert np.array_equal(e.labels(), lab)
        e.close()


def test_encode_and_relabel_reuse_their_memory():
    e = L.Engine(0)
    for scale in (17, 12, 19, 12, 17):
        g = L.gen_rmat(scale, 16, seed=scale, bfs=False)
        row, col, perm = e.bfs_relabel(g.row, g.col, 0)
        h, hperm = g.bfs_relabel(0)
        assert np.array_equal(perm, hperm) and np.array_equal(row, h.row) and np.array_equal(col, h.col)
        for T in (0, 16):
            cgr = h.encode(T, 128)
            e.encode_csr(row, col, T)
            words, offs, vert, nbits = e.stream()
            assert nbits == cgr.nbits and np.array_equal(offs, cgr.offsets) and np.array_equal(vert, cgr.vertices)
            host = np.frombuffer(cgr.stream_bytes(), np.uint8)
            assert np.array_equal(words.astype(">u8").view(np.uint8)[:len(host)], host)
    e.close()
