"""The LDS window reader of cgr_decode.hpp, built for the host, against the
oracle: golden and generated streams, codes longer than 32 bits, and records
of which only the first words are staged."""
import ctypes as C
import os

import numpy as np
import pytest

import lpa_amd as L
import pyoracle as O
from helpers import golden_cases, load_golden
from test_device_decoder_host import words64

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "libdecode_check.so")


@pytest.fixture(scope="module")
def dc():
    lib = C.CDLL(LIB)
    P = C.c_void_p
    lib.dc_decode_record_window.restype = C.c_int64
    lib.dc_decode_record_window.argtypes = [P, C.c_uint64, C.c_uint64, C.c_uint32, P, C.c_uint64, C.c_int, C.c_uint64]
    return lib


def check(dc, stream, nbits, starts, vertices, step=1):
    w = words64(stream)
    raw = np.frombuffer(bytes(stream), np.uint8)
    cap = 1 << 16
    out = np.zeros(cap, np.uint32)
    for i in range(0, len(starts) - 1, step):
        v, a, b = int(vertices[i]), int(starts[i]), int(starts[i + 1])
        want, _ = O.decode_record(raw, nbits, a, v, cap=cap)
        for chk, have in ((0, 0), (1, 1), (1, 3), (1, 1 << 30)):
            d = dc.dc_decode_record_window(w.ctypes.data, a, b, v, out.ctypes.data, cap, chk, have)
            assert d == len(want) and np.array_equal(out[:d], want), (i, v, chk, have)


@pytest.mark.parametrize("case", golden_cases())
def test_golden(dc, case):
    g = load_golden(case)
    starts = np.concatenate([[0], g["end_offs"]]).astype(np.uint64)
    check(dc, g["stream"], int(g["end_offs"][-1]) if g["n_c"] else 0, starts, g["vertices"])


@pytest.mark.parametrize("gen", ["rmat", "lattice", "copying"])
def test_generated(dc, gen):
    g = {"rmat": lambda: L.gen_rmat(13, 16, seed=7), "lattice": lambda: L.gen_lattice(64, 0.1, 0.005, seed=1),
         "copying": lambda: L.gen_copying(8000, 30.0, 2.1, 4000, 0.7, 200, seed=3)}[gen]()
    c = g.encode(0, 128)
    check(dc, c.stream_bytes(), c.nbits, c.offsets, c.vertices, step=3)


def test_long_codes(dc):
    """gaps and first codes around the 32-bit limits of the fast paths: gamma
    of 2^16 - 1, zeta of 2^24 - 1, up to ids near 2^30"""
    n = (1 << 30) - 1
    rng = np.random.default_rng(0)
    rows = []
    for edge in (1 << 14, 1 << 15, 1 << 16, 1 << 23, 1 << 24, 1 << 27, 1 << 29):
        for delta in (-3, -2, -1, 0, 1, 2):
            g = edge + delta
            rows.append(np.array([g, 2 * g if 2 * g < n else g + 1], np.int64))
            run = np.arange(4)
            rows.append(np.concatenate([run + 5, run + 9 + g] if 9 + g + 4 < n else [run + 5]))
    rows.append(np.sort(rng.choice(n, 300, replace=False)))
    rows.append(np.arange(70_000))          # one interval whose length takes a long gamma
    for v in (0, 1 << 20, n - 1):
        words, starts = [], [0]
        lib = dc
        lib.dc_encode_bits.restype = C.c_uint64
        lib.dc_encode_bits.argtypes = [C.c_uint32, C.c_void_p, C.c_uint32]
        lib.dc_encode_record.restype = None
        lib.dc_encode_record.argtypes = [C.c_uint32, C.c_void_p, C.c_uint32, C.c_void_p, C.c_uint64, C.c_uint64]
        adj = [np.ascontiguousarray(r, np.uint32) for r in rows]
        for a in adj:
            starts.append(starts[-1] + lib.dc_encode_bits(v, a.ctypes.data, len(a)))
        words = np.zeros(starts[-1] // 64 + 10, np.uint64)
        for a, s, e in zip(adj, starts, starts[1:]):
            lib.dc_encode_record(v, a.ctypes.data, len(a), words.ctypes.data, s, e)
        out = np.zeros(1 << 17, np.uint32)
        for a, s, e in zip(adj, starts, starts[1:]):
            for chk, have in ((0, 0), (1, 2)):
                d = lib.dc_decode_record_window(words.ctypes.data, s, e, v, out.ctypes.data, 1 << 17, chk, have)
                # intervals come before residuals: compare as sets of ids
                assert d == len(a) and np.array_equal(np.sort(out[:d]), a), (v, len(a), a[:2], chk)
