"""Device encoding of rows around the limits of the lane (16 ids), wave and
workgroup (8192 ids) encoders and of the wave's 64-id rounds: the stream is
the host encoder's, bit for bit, with and without the allocating entry
point's workgroup kernels."""
import numpy as np
import pytest

import lpa_amd as L
from test_zz_no_alloc import encode_no_alloc

pytestmark = pytest.mark.gpu

N = 150_000
DEGREES = [1, 15, 16, 17, 18, 62, 63, 64, 65, 66, 67, 127, 128, 129, 130, 191, 192, 193, 320, 1000, 8191, 8192, 8193,
           9000]


def _row(kind, d, rng):
    if kind == "singles":                       # no interval
        ids = np.arange(d) * 3
    elif kind == "one_run":                     # one interval over every round
        ids = np.arange(d)
    elif kind == "threes_and_fours":            # runs that just miss, just make an interval
        run = np.arange(d)
        ids = run + 2 * (run // 7) + (run % 7 >= 3) * 2
    elif kind == "dense":                       # 4-bit codes: the fullest segments
        ids = np.arange(d) * 2
    else:                                       # runs of any length, gaps up to thousands
        gaps = np.where(rng.random(d) < 0.7, 1, rng.integers(2, 12, d))
        gaps[rng.random(d) < 0.01] = 3000
        ids = np.cumsum(gaps)
    off = int(rng.integers(0, max(1, N - int(ids[-1]) - 1))) if ids[-1] < N - 1 else 0
    ids = ids + off
    return ids[ids < N].astype(np.uint32)


def _graph(kind):
    rng = np.random.default_rng(len(kind))
    rows = [np.zeros(0, np.uint32)] * N
    for i, d in enumerate(DEGREES * 3):
        rows[int(rng.integers(0, N - 1)) if i % 3 else i * 1000] = _row(kind, d, rng)
    row = np.zeros(N + 1, np.uint64)
    row[1:] = np.cumsum([len(r) for r in rows])
    return L.Csr.from_arrays(row, np.concatenate(rows))


@pytest.mark.parametrize("kind", ["singles", "one_run", "threes_and_fours", "dense", "mixed"])
def test_rows_around_the_limits(kind):
    g = _graph(kind)
    cgr = g.encode(0, 128)
    e = L.Engine(0)
    e.encode_csr(g.row, g.col, 0)
    words, offs, vert, nbits = e.stream()
    assert nbits == cgr.nbits and np.array_equal(offs, cgr.offsets) and np.array_equal(vert, cgr.vertices)
    host = np.frombuffer(cgr.stream_bytes(), np.uint8)
    raw = words.astype(">u8").view(np.uint8)
    assert np.array_equal(raw[:len(host)], host)
    # degrees and features come from the validation pass over these records
    assert np.array_equal(e.degrees(), np.diff(g.row.astype(np.int64)))
    rc, offs2, words2, nbits2 = encode_no_alloc(e, g.row, g.col, 0)
    assert rc == 0 and nbits2 == nbits and np.array_equal(offs2, offs) and np.array_equal(words2, words)
    e.close()


@pytest.mark.parametrize("d", [17, 64, 65, 8193])
def test_bad_rows_are_rejected(d):
    for where, value in ((d // 2, None), (d - 1, N)):   # a repeated id; an id >= n
        col = (np.arange(d) * 2).astype(np.uint32)
        col[where] = col[where - 1] if value is None else value
        row = np.zeros(N + 1, np.uint64)
        row[5:] = d
        e = L.Engine(0)
        with pytest.raises(L.LpaError):
            e.encode_csr(row, col, 0)
        e.close()


def test_more_rows_than_one_launch_holds():
    """2^26 rows are 2^32 threads at a wave each: several launches, with rows
    for the wave encoder at both sides of every joint and at the end"""
    n = (1 << 26) + 70
    d = np.zeros(n, np.int64)
    for at in (0, (1 << 25) - 1, 1 << 25, (1 << 26) - 1, 1 << 26, n - 1):
        d[at] = 40
    row = np.zeros(n + 1, np.uint64)
    np.cumsum(d, out=row[1:].view(np.int64))
    col = np.concatenate([np.arange(40, dtype=np.uint32) * (3 + i) + i for i in range(6)])
    g = L.Csr.from_arrays(row, col)
    cgr = g.encode(0, 128)
    e = L.Engine(0)
    e.encode_csr(g.row, g.col, 0)
    words, offs, _, nbits = e.stream()
    assert nbits == cgr.nbits and np.array_equal(offs, cgr.offsets)
    host = np.frombuffer(cgr.stream_bytes(), np.uint8)
    assert np.array_equal(words.astype(">u8").view(np.uint8)[:len(host)], host)
    deg = e.degrees()
    assert np.array_equal(deg, d)
