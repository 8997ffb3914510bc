"""More products at once than a launch has rows for their transforms: a slab
of 40,000 residues and a batch of 33,000 pairs of one size, compared with the
oracle at the edges of the parts and in between.  Bit-exact."""
import ctypes as C

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
P = C.POINTER(C.c_uint64)


@pytest.fixture(scope="module", autouse=True)
def dev():
    from mersenne_trinomial_amd import device
    device.init(0)


def rand_bits(rng, n, bits, pitch):
    a = np.zeros((n, pitch), np.uint64)
    a[:, :O.words(bits)] = rng.integers(0, 2**64, (n, O.words(bits)), dtype=np.uint64)
    if bits & 63:
        a[:, O.words(bits) - 1] &= np.uint64((1 << (bits & 63)) - 1)
    return a


def test_slab():
    from mersenne_trinomial_amd._capi import check, lib
    from mersenne_trinomial_amd.device import DeviceBuffer
    r, n = 9001, 40000
    nw = O.words(r)
    pitch = nw + 3
    rng = np.random.default_rng(1)
    a, b = rand_bits(rng, n, r, pitch), rand_bits(rng, n, r, pitch)
    s = rng.integers(1, (r - 1) // 2 + 1, n, dtype=np.uint64)
    A, B, S = DeviceBuffer.from_array(a), DeviceBuffer.from_array(b), DeviceBuffer.from_array(s)
    work = DeviceBuffer(lib.gf2t_mulmod_slab_workspace_bytes(r, n))
    check(lib.gf2t_mulmod_slab(A.ptr, pitch, B.ptr, pitch, 1, r, S.ptr, A.ptr, pitch, n, work.ptr,
                               None))
    got = A.download().reshape(n, pitch)
    for i in [0, 1, 32765, 32766, 32767, 32768, n - 1] + list(rng.integers(0, n, 50)):
        t = b[i, :nw].copy()
        t[0] ^= np.uint64(2)
        assert np.array_equal(got[i, :nw], O.mulmod(a[i, :nw].copy(), r, t, r, r, int(s[i]))), i


def test_batch():
    from mersenne_trinomial_amd._capi import check, lib
    from mersenne_trinomial_amd.device import DeviceBuffer
    r, n, bits, few = 20011, 33000, 20000, 7
    nw, bw = O.words(r), O.words(bits)
    rng = np.random.default_rng(2)
    a, b = rand_bits(rng, few, bits, bw), rand_bits(rng, few, bits, bw)
    s = rng.integers(1, (r - 1) // 2 + 1, n, dtype=np.uint64)
    A, B, out = DeviceBuffer.from_array(a), DeviceBuffer.from_array(b), DeviceBuffer.words(n * nw)
    ptrs = lambda v: (C.c_void_p * n)(*v)
    pa = ptrs([A.ptr + 8 * bw * (j % few) for j in range(n)])
    pb = ptrs([B.ptr + 8 * bw * (j // few % few) for j in range(n)])
    po = ptrs([out.ptr + 8 * nw * j for j in range(n)])
    nb = np.full(n, bits, np.uint64)
    p = lambda v: v.ctypes.data_as(P)
    work = DeviceBuffer(lib.gf2t_mulmod_batch_workspace_bytes(n, p(nb), p(nb)))
    check(lib.gf2t_mulmod_batch(n, pa, p(nb), pb, p(nb), r, p(s), po, work.ptr, None))
    got = out.download().reshape(n, nw)
    for j in [0, 1, 32766, 32767, 32768, n - 1] + list(rng.integers(0, n, 50)):
        want = O.mulmod(a[j % few], bits, b[j // few % few], bits, r, int(s[j]))
        assert np.array_equal(got[j], want), j
