"""The Cantor transform's emulation (test_cantor_logic.py) at a size where the
low levels of a transform by itself take twiddles of GF(2^32), and single
tiles of the butterfly windows of larger transforms, whose twiddles lie there
from 2^25 points on, against GF(2^64) products.  No GPU."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import oracle as O
from test_cantor_logic import CSRC, HERE, P64, cl  # noqa: F401


def test_transform_low_levels_32(cl):  # noqa: F811
    m = 23
    rng = np.random.default_rng(m)
    f = rng.integers(0, 2**64, 1 << m, dtype=np.uint64)
    g = f.copy()
    cl.cl_fft(g.ctypes.data_as(P64), m, 0, 13, 12, 10)
    assert np.array_equal(g, O.fft_fwd(f, m))
    cl.cl_fft(g.ctypes.data_as(P64), m, 1, 13, 12, 10)
    assert np.array_equal(g, f)


@pytest.fixture(scope="module")
def cw(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("cw") / "libcw.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I" + CSRC, "-o", out,
                           os.path.join(HERE, "host", "cantor_windows.cpp")])
    lib = C.CDLL(out)
    lib.cw_check.argtypes = [P64] + [C.c_int] * 3 + [C.c_uint64, C.c_int, C.c_void_p]
    return lib


@pytest.mark.parametrize("m", [9, 17, 24, 25, 26, 27])
def test_windows(cw, m):
    b, rng, cls = O.cantor_basis(), np.random.default_rng(m), C.c_int()
    seen = set()
    for tile_bits in (10, 8):
        for p in range(3):
            for blk in [0, 1, 2**31 - 1] + [int(x) for x in rng.integers(0, 2**31, 5)]:
                for inv in (0, 1):
                    got = cw.cw_check(b.ctypes.data_as(P64), m, tile_bits, p, blk, inv, C.addressof(cls))
                    assert got == (0 if p < (m - 1) // 8 else -1), (tile_bits, p, blk, inv)
                    seen.add(cls.value)
    assert (32 in seen) == (m >= 25)
