"""Products at the edges of their launch rules, against the oracle: without a
transform (tiles of 128 chunks, one product or nine of a quarter, few and
many parts, unbalanced operands, the largest), the transforms' sizes whose
twiddle classes and windows change, and batches of mixed sizes.  Bit-exact."""
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
    a = rng.integers(0, 2**64, (bits + 63) // 64, dtype=np.uint64)
    if bits & 63:
        a[-1] &= np.uint64((1 << (bits & 63)) - 1)
    return a


def same(got, want):
    n = max(got.size, want.size)
    return np.array_equal(np.pad(got, (0, n - got.size)), np.pad(want, (0, n - want.size)))


# chunks of the operands
@pytest.mark.parametrize("ca,cb", [(1, 1), (127, 128), (128, 129), (129, 129), (129, 1000), (511, 511),
                                   (511, 512), (512, 512), (513, 515), (512, 513), (514, 4000), (639, 640),
                                   (1021, 2050), (1023, 1024), (1024, 1024), (2047, 2049), (3, 40000), (700, 64000), (10239, 10240), (10240, 10241)])
def test_product_without_transform(eng, ca, cb):
    rng = np.random.default_rng(ca * 65537 + cb)
    abits, bbits = 32 * ca - int(rng.integers(0, 32)), 32 * cb - int(rng.integers(0, 32))
    a, b = rand_bits(rng, abits), rand_bits(rng, bbits)
    want = O.fft_mul(a, abits, b, bbits)
    assert same(eng.mul(a, abits, b, bbits), want)
    assert same(eng.mul(b, bbits, a, abits), want)


@pytest.mark.parametrize("r,s", [(4096 * 4, 5), (16383, 8000), (16385, 1), (32736, 177), (32737, 177), (65537, 32768)])
def test_mulmod_without_transform(eng, r, s):
    rng = np.random.default_rng(r)
    a, b = rand_bits(rng, r), rand_bits(rng, r)
    assert np.array_equal(eng.mulmod(a, r, b, r, r, s), O.mulmod(a, r, b, r, r, s))


# 2^m points, at the least and the most chunks of each
@pytest.mark.parametrize("m", [15, 16, 17, 18, 19, 20])
@pytest.mark.parametrize("most", [False, True])
def test_transform_sizes(eng, m, most):
    rng = np.random.default_rng(2 * m + most)
    total = (1 << m) + 1 if most else (1 << (m - 1)) + 2   # chunks of both operands
    ca = max(1, total // 3)
    abits, bbits = 32 * ca - 7, 32 * (total - ca)
    a, b = rand_bits(rng, abits), rand_bits(rng, bbits)
    assert same(eng.mul(a, abits, b, bbits), O.fft_mul(a, abits, b, bbits))


def test_batch_of_mixed_sizes(eng):
    """Pairs shorter and longer than a block's run of the grouped passes,
    empty ones among them."""
    import ctypes as C
    from mersenne_trinomial_amd._capi import check, lib
    from mersenne_trinomial_amd.device import DeviceBuffer
    r, s = 132049, [1, 66024, 500, 7, 32768, 90, 3]
    bits = [(132049, 132049), (40, 132049), (65536, 65537), (0, 100), (131072, 64), (1, 1), (90000, 132049)]
    rng = np.random.default_rng(3)
    a = [rand_bits(rng, max(x, 1)) for x, _ in bits]
    b = [rand_bits(rng, max(y, 1)) for _, y in bits]
    n, P = len(bits), C.POINTER(C.c_uint64)
    A, B = [DeviceBuffer.from_array(x) for x in a], [DeviceBuffer.from_array(x) for x in b]
    out = [DeviceBuffer.words(O.words(r)) for _ in range(n)]
    ab, bb, ss = (np.array(v, dtype=np.uint64) for v in ([x for x, _ in bits], [y for _, y in bits], s))
    p = lambda v: v.ctypes.data_as(P)
    work = DeviceBuffer(lib.gf2t_mulmod_batch_workspace_bytes(n, p(ab), p(bb)))
    ptrs = lambda l: (C.c_void_p * n)(*[x.ptr for x in l])
    check(lib.gf2t_mulmod_batch(n, ptrs(A), p(ab), ptrs(B), p(bb), r, p(ss), ptrs(out), work.ptr, None))
    for k, (x, y) in enumerate(bits):
        want = O.mulmod(a[k], x, b[k], y, r, s[k]) if x and y else np.zeros(O.words(r), np.uint64)
        assert np.array_equal(out[k].download(O.words(r)), want), k
