"""Decoding from staged words: degrees around the kernels' limits, the decoded
CSR's rows, and streams whose segments are nearly empty, so that a record or a
workgroup's records outgrow the staging memory and are read in place."""
import numpy as np
import pytest

import lpa_amd as L
import pyoracle as O

pytestmark = pytest.mark.gpu

DEGREES = [1, 4, 5, 8, 9, 16, 17, 32, 33, 64, 65, 128, 129, 256, 257, 512, 513, 1024, 1025, 2048, 2049, 4096, 4097, 9000]
N = 30_000


def _csr(kind):
    rng = np.random.default_rng(3)
    rows = [np.zeros(0, np.uint32)] * N
    for i, d in enumerate(DEGREES * 4):
        if kind == "residuals":
            ids = np.sort(rng.choice(N, d, replace=False))
        else:                                   # short and long runs
            ids = np.unique(np.concatenate([np.arange(s, s + r) for s, r in
                                            zip(rng.integers(0, N - 400, d // 6 + 1), rng.integers(1, 40, d // 6 + 1))]))[:d]
        rows[i * 300 + i % 7] = ids.astype(np.uint32)
    row = np.zeros(N + 1, np.uint64)
    row[1:] = np.cumsum([len(r) for r in rows])
    return row, np.concatenate(rows)


def _steps(e, row, col, K, method, iters=3):
    e.config(K=K)
    e.schedule_degree()
    e.labels_init()
    c = O.cfg(K=K)
    lab = np.repeat(np.arange(len(row) - 1, dtype=np.uint32), K)
    for _ in range(iters):
        ch = {"nova": e.nova_iterate, "cglp": e.cglp_iterate}[method]()
        lab, och = O.step_csr(row, col, lab, c)
        assert ch == och and np.array_equal(e.labels(), lab)


def _check_rows(e, row, col):
    got_row, got = e.cglp_csr()
    assert np.array_equal(got_row, row)
    for v in np.nonzero(np.diff(row.astype(np.int64)))[0]:
        a, b = int(row[v]), int(row[v + 1])
        assert np.array_equal(np.sort(got[a:b]), col[a:b]), v


@pytest.mark.parametrize("kind", ["residuals", "runs"])
@pytest.mark.parametrize("K", [1, 5])
def test_degrees_around_the_limits(kind, K):
    row, col = _csr(kind)
    e = L.Engine(0)
    e.upload(L.Csr.from_arrays(row, col).encode(0, 128))
    _steps(e, row, col, K, "nova")
    _steps(e, row, col, K, "cglp")
    _check_rows(e, row, col)
    e.close()


def _gamma(x):
    b = bin(x + 1)[2:]
    return "0" * (len(b) - 1) + b


def _zeta(x):
    h = ((x + 1).bit_length() - 1) // 3
    return "0" * h + "1" + format(x + 1, f"0{3 * (h + 1)}b")


def _loose_record(v, ids):
    """every residual segment holds one id: 256 bits each"""
    out = _gamma(0) + _gamma(0)
    segs = []
    for u in ids:
        d = int(u) - v
        segs.append(_gamma(1) + _zeta(2 * d if d >= 0 else -2 * d - 1))
    if not segs:
        return out + _gamma(0) + _gamma(0)
    return out + _gamma(len(segs) - 1) + "".join(s.ljust(256, "0") for s in segs[:-1]) + segs[-1]


def test_loosely_packed_stream():
    rng = np.random.default_rng(5)
    n = 3000
    rows = [np.sort(rng.choice(n, int(d), replace=False)).astype(np.uint32)
            for d in rng.choice([0, 1, 3, 4, 7, 16, 31, 60, 120, 300, 700, 3000], n, p=[.3, .1, .1, .1, .1, .1, .1, .04, .03, .02, .009, .001])]
    order = np.array([v for v in range(n) if len(rows[v]) >= 128] + [v for v in range(n) if len(rows[v]) < 128], np.uint32)
    bits = [_loose_record(int(v), rows[v]) for v in order]
    offs = np.concatenate([[0], np.cumsum([len(b) for b in bits])]).astype(np.uint64)
    s = "".join(bits)
    s += "0" * (-len(s) % 32)
    words = np.frombuffer(int(s, 2).to_bytes(len(s) // 8, "big"), ">u4").astype(np.uint32)
    row = np.zeros(n + 1, np.uint64)
    row[1:] = np.cumsum([len(r) for r in rows])
    col = np.concatenate(rows)
    e = L.Engine(0)
    e.upload_arrays(n, n, words, len(words), offs, order)
    assert np.array_equal(e.degrees(), np.diff(row.astype(np.int64)))
    for K in (1, 8):
        _steps(e, row, col, K, "nova")
    _steps(e, row, col, 1, "cglp")
    _check_rows(e, row, col)
    e.close()
