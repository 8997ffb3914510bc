"""Products whose tiles are mostly empty, at the edges of what k_school skips
(a wave's 32 values, half a tile's 64 outputs, a tile's 128), and slabs on
both sides of the lines between that kernel and transforms, against the
oracle.  Bit-exact."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    import mersenne_trinomial_amd as M
    from mersenne_trinomial_amd import device
    device.init(0)
    return M


def rand_bits(rng, bits):
    a = rng.integers(0, 2**64, O.words(bits), dtype=np.uint64)
    if bits & 63:
        a[-1] &= np.uint64((1 << (bits & 63)) - 1)
    return a


# chunks of the operands
@pytest.mark.parametrize("ca,cb", [(1, 1), (1, 64), (1, 129), (2, 130), (31, 33), (32, 32), (33, 32), (63, 64), (64, 65),
                                   (65, 200), (96, 96), (97, 127), (100, 1000), (127, 127), (128, 300), (129, 64),
                                   (130, 130), (160, 161), (193, 256), (300, 1023)])
def test_product_and_fold(eng, ca, cb):
    rng = np.random.default_rng(1000 * ca + cb)
    abits, bbits = 32 * ca - int(rng.integers(0, 32)), 32 * cb - int(rng.integers(0, 32))
    a, b = rand_bits(rng, abits), rand_bits(rng, bbits)
    want = O.mul_comb(a, abits, b, bbits)
    for x, xb, y, yb in ((a, abits, b, bbits), (b, bbits, a, abits)):
        got = eng.mul(x, xb, y, yb)
        n = max(got.size, want.size)
        assert np.array_equal(np.pad(got, (0, n - got.size)), np.pad(want, (0, n - want.size)))
        r = max(3, (abits + bbits + 1) // 2, abits, bbits)
        assert np.array_equal(eng.mulmod(x, xb, y, yb, r, 1), O.mulmod(x, xb, y, yb, r, 1))


@pytest.mark.parametrize("r,n", [(5, 3), (31, 2), (89, 1000), (1025, 3), (2047, 3), (3071, 40), (4096, 5), (4097, 5),
                                 (4423, 868), (4423, 869), (8192, 3)])
def test_slab(eng, r, n):
    from mersenne_trinomial_amd._capi import check, lib
    from mersenne_trinomial_amd.device import DeviceBuffer
    nw = O.words(r)
    pitch = nw + 1
    rng = np.random.default_rng(r + n)
    a, b = (np.zeros((n, pitch), np.uint64) for _ in range(2))
    for v in (a, b):
        v[:, :nw] = rng.integers(0, 2**64, (n, nw), dtype=np.uint64)
        if r & 63:
            v[:, nw - 1] &= np.uint64((1 << (r & 63)) - 1)
    s = rng.integers(1, (r - 1) // 2 + 1, n, dtype=np.uint64)
    A, B, S = DeviceBuffer.from_array(a), DeviceBuffer.from_array(b), DeviceBuffer.from_array(s)
    out, work = DeviceBuffer.words(n * pitch), DeviceBuffer(lib.gf2t_mulmod_slab_workspace_bytes(r, n))
    for add_x in (0, 1):
        check(lib.gf2t_mulmod_slab(A.ptr, pitch, B.ptr, pitch, add_x, r, S.ptr, out.ptr, pitch, n, work.ptr, None))
        got = out.download().reshape(n, pitch)
        for i in sorted({0, n // 2, n - 1}):
            t = b[i, :nw].copy()
            t[0] ^= np.uint64(2 * add_x)
            assert np.array_equal(got[i, :nw], O.mulmod(a[i, :nw].copy(), r, t, r, r, int(s[i]))), (add_x, i)
