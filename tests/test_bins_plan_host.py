"""Launch plans of the group kernels on the host: for every schedule that a
caller may ask for, the LDS that a launch is given holds what its kernel
addresses, by itself and merged with other bins, and a merged bin always
reaches a kernel that the merged launch has."""
import ctypes as C
import os

import numpy as np
import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "libbins_check.so")


@pytest.fixture(scope="module")
def bc():
    lib = C.CDLL(LIB)
    lib.bc_plan.argtypes = [C.c_uint32, C.c_uint32, C.c_uint32, C.c_int, C.c_int, C.c_void_p]
    lib.bc_plan.restype = None
    return lib


QUARTER = [0, 1, 16, 32, 33, 63, 64, 65, 100, 127, 128, 129, 200, 255, 256, 257, 300, 511, 512, 513, 1024, 1 << 31]


@pytest.mark.parametrize("K", list(range(1, 10)) + [16, 17, 33, 64])
def test_lds_given_holds_lds_addressed(bc, K):
    out = np.zeros(7, np.uint64)
    merged = 0
    for block, logts in ((0, range(6, 12)), (1, range(8, 14))):
        for q in QUARTER:
            for logt in logts:
                for csr in (0, 1):
                    bc.bc_plan(K, q, logt, block, csr, out.ctypes.data)
                    ng, ids, given, used, held, m_given, m_used = (int(x) for x in out)
                    where = dict(K=K, quarter_max=q, logT=logt, block=block, csr=csr, groups=ng, ids=ids)
                    assert used <= given, where
                    if held:
                        merged += 1
                        assert m_used <= m_given, where
                        assert bc.bc_held(1 if K == 1 else 2 if K == 2 else 4 if K <= 4 else 8, 256 // ng, ids), where
    assert merged


def test_unusual_half_waves_are_launched_alone(bc):
    """129 to 256 ids in half waves: 8 staged ids per lane, which the merged
    kernel of 8 vectors does not have"""
    out = np.zeros(7, np.uint64)
    for K in (5, 6, 7, 8, 9, 64):
        bc.bc_plan(K, 256, 9, 0, 0, out.ctypes.data)
        assert out[0] == 8 and out[1] == 8 and out[4] == 0
        bc.bc_plan(K, 128, 8, 0, 0, out.ctypes.data)
        assert out[0] == 8 and out[1] == 4 and out[4] == 1
