"""Matrix-vector products of the host service without transforms: single
chunks, zero entries, entries shorter and longer than the vectors, one to four
pairs, operands read in place and copied, and both sides of the line to
transforms, against the oracle.  Bit-exact."""
import ctypes as C

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
P = C.POINTER(C.c_uint64)


def rand(rng, bits):
    v = rng.integers(0, 2**64, max(1, O.words(bits)), dtype=np.uint64)
    if bits & 63:
        v[-1] &= np.uint64((1 << (bits & 63)) - 1)
    return v if bits else np.zeros(1, np.uint64)


# bits of the matrix' entries, and of the vectors'
@pytest.mark.parametrize("mbits,vbits", [((1, 1, 1, 1), (1, 33)), ((64, 0, 5, 31), (2000, 1, 0, 1999)),
                                         ((4096, 4095, 4000, 0), (4096, 77) * 2), ((9000, 8000, 1, 70), (300, 299)),
                                         ((16000,) * 4, (16383, 16384) * 4), ((46305, 46300, 32, 40000), (46305, 46000) * 4),
                                         ((46400,) * 4, (46400, 46399) * 4), ((3000, 2999, 3000, 2000), (200000, 100))])
@pytest.mark.parametrize("zc", [0, 65536])
def test_mat2n(mbits, vbits, zc):
    from mersenne_trinomial_amd import device
    from mersenne_trinomial_amd._capi import check, lib
    device.init(0)
    rng = np.random.default_rng(len(vbits) + sum(mbits))
    m, v = [rand(rng, b) for b in mbits], [rand(rng, b) for b in vbits]
    n = len(v) // 2
    ow = int(lib.gf2t_mul_out_words(max(mbits), max(vbits))) + 2
    out = [np.full(ow, 7, np.uint64) for _ in v]
    ptrs = lambda l: (P * len(l))(*[x.ctypes.data_as(P) for x in l])
    U = lambda l: (C.c_uint64 * len(l))(*l)
    old = C.c_int64()
    check(lib.gf2t_tune_get(b"hm_zc_words", C.byref(old)))
    check(lib.gf2t_tune(b"hm_zc_words", zc))
    try:
        check(lib.gf2t_mat2n_host(ptrs(m), U(mbits), n, ptrs(v), U(vbits), ptrs(out), ow))
    finally:
        check(lib.gf2t_tune(b"hm_zc_words", old.value))
    for p in range(n):
        for o in range(2):
            want = np.zeros(ow, np.uint64)
            for h in range(2):
                a, b = mbits[2 * o + h], vbits[2 * p + h]
                if a and b:
                    w = O.fft_mul(m[2 * o + h], a, v[2 * p + h], b)
                    want[:w.size] ^= w
            assert np.array_equal(out[2 * p + o], want), (p, o)
