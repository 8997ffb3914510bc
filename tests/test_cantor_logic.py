"""The Cantor transform's tables, index maps and arithmetic (cantor.hpp,
shared with the gfx950 kernels) emulated thread by thread on the host and
checked against the oracle.  No GPU."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import oracle as O

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "mersenne_trinomial_amd", "csrc")
P64, P32 = C.POINTER(C.c_uint64), C.POINTER(C.c_uint32)


@pytest.fixture(scope="module")
def cl(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("cl") / "libcl.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I" + CSRC, "-o", out,
                           os.path.join(HERE, "host", "cantor_logic.cpp")])
    lib = C.CDLL(out)
    lib.cl_fft.argtypes = [P64] + [C.c_int] * 5
    lib.cl_product.argtypes = [P32, C.c_size_t, P32, C.c_size_t, C.c_int, P64] + [C.c_int] * 3
    b = O.cantor_basis()
    assert lib.cl_init(b.ctypes.data_as(P64)) == 0
    return lib


# every size to 2^18 (windows of one to eight bits above the low eight, one
# and two of them, every subfield class); 20 and 25 for the third
# window's shapes at smaller tiles
@pytest.mark.parametrize("m", list(range(1, 19)) + [20])
@pytest.mark.parametrize("one,tb,bf", [(13, 13, 10), (12, 12, 8)])
def test_transform(cl, m, one, tb, bf):
    rng = np.random.default_rng(m)
    f = rng.integers(0, 2**64, 1 << m, dtype=np.uint64)
    g = f.copy()
    cl.cl_fft(g.ctypes.data_as(P64), m, 0, one, tb, bf)
    assert np.array_equal(g, O.fft_fwd(f, m))
    cl.cl_fft(g.ctypes.data_as(P64), m, 1, one, tb, bf)
    assert np.array_equal(g, f)


@pytest.mark.parametrize("na,nb", [(1, 1), (2, 3), (5, 4), (129, 128), (300, 213), (4097, 1),
                                   (4096, 4097), (5000, 3193), (33000, 70)])
def test_product(cl, na, nb):
    rng = np.random.default_rng(na + 7 * nb)
    a = rng.integers(0, 2**32, na, dtype=np.uint32)
    b = rng.integers(0, 2**32, nb, dtype=np.uint32)
    m = 1
    while (1 << m) < na + nb - 1:
        m += 1
    out = np.zeros(1 << m, np.uint64)
    cl.cl_product(a.ctypes.data_as(P32), na, b.ctypes.data_as(P32), nb, m,
                  out.ctypes.data_as(P64), 13, 13, 10)
    lo, hi = (out & np.uint64(0xFFFFFFFF)).astype(np.uint32), (out >> np.uint64(32)).astype(np.uint32)
    got = np.zeros(na + nb + 1, np.uint32)
    n = min(out.size, got.size - 1)
    got[:n] ^= lo[:n]
    got[1:n + 1] ^= hi[:n]

    def words(x):
        return np.concatenate([x, np.zeros(x.size & 1, np.uint32)]).view(np.uint64)
    want = O.fft_mul(words(a), 32 * na, words(b), 32 * nb)
    assert np.array_equal(words(got)[:want.size], want[:words(got).size])
