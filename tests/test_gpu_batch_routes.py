"""Batches of products by their routes: all without transforms (very unequal
operands, one chunk, single words of output, zero operands among them), none,
and sizes on both sides of the line between the two, against the oracle.
Bit-exact."""
import ctypes as C

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

BATCHES = {
    "one": (132049, [(132049, 132049)]),
    "tiny": (67, [(67, 67), (1, 67), (32, 33), (3, 5), (0, 67), (64, 64)] * 50),
    "unequal": (400000, [(32, 399000), (64, 399990), (33, 1), (5000, 200000), (1, 400000), (4097, 131000)]),
    "sizes": (132049, [(1 << k, (1 << k) - 3) for k in range(5, 17)]),
    "line": (262145, [(40, 50), (262144, 262144), (1024, 999), (131072, 131072), (262144, 100), (65536, 131072),
                      (7, 262145), (131073, 131072), (100000, 150000)]),
    "large": (1 << 21, [(1 << 21, 1 << 20), (1 << 20, (1 << 20) + 3), (1 << 21, 5)]),
}


@pytest.mark.parametrize("name", list(BATCHES))
def test_batch(name):
    from mersenne_trinomial_amd import device
    from mersenne_trinomial_amd._capi import check, lib
    from mersenne_trinomial_amd.device import DeviceBuffer
    device.init(0)
    r, bits = BATCHES[name]
    bits = [(a, min(b, 2 * r - a)) for a, b in bits]
    rng = np.random.default_rng(len(bits) + r)

    def rand(k):
        v = rng.integers(0, 2**64, max(1, O.words(k)), dtype=np.uint64)
        if k & 63:
            v[-1] &= np.uint64((1 << (k & 63)) - 1)
        return v
    a, b = [rand(x) for x, _ in bits], [rand(y) for _, y in bits]
    s = [int(v) for v in rng.integers(1, (r - 1) // 2 + 1, len(bits))]
    n, P = len(bits), C.POINTER(C.c_uint64)
    A, B = [DeviceBuffer.from_array(x) for x in a], [DeviceBuffer.from_array(x) for x in b]
    out = [DeviceBuffer.words(O.words(r)) for _ in range(n)]
    ab, bb, ss = (np.array(v, dtype=np.uint64) for v in ([x for x, _ in bits], [y for _, y in bits], s))
    p, ptrs = lambda v: v.ctypes.data_as(P), lambda l: (C.c_void_p * n)(*[x.ptr for x in l])
    work = DeviceBuffer(lib.gf2t_mulmod_batch_workspace_bytes(n, p(ab), p(bb)))
    check(lib.gf2t_mulmod_batch(n, ptrs(A), p(ab), ptrs(B), p(bb), r, p(ss), ptrs(out), work.ptr, None))
    for k, (x, y) in enumerate(bits):
        want = O.mulmod(a[k], x, b[k], y, r, s[k]) if x and y else np.zeros(O.words(r), np.uint64)
        assert np.array_equal(out[k].download(), want), (k, x, y)
