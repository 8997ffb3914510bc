"""Wrapped products (2^mp + e coefficients by 2^mp-point transforms and a
product of the top chunks) on both sides of their rule, against the oracle.
Bit-exact."""
import numpy as np
import pytest

import oracle as O
import wrapped_shapes as W

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


@pytest.mark.parametrize("mp,e,ca,on", W.PRODUCTS)
def test_product(eng, mp, e, ca, on):
    rng = np.random.default_rng(mp + e + ca)
    abits, bbits = 32 * ca - int(rng.integers(0, 32)), 32 * W.other(mp, e, ca) - int(rng.integers(0, 32))
    a, b = rand_bits(rng, abits), rand_bits(rng, bbits)
    print(f"2^{mp} + {e} coefficients: {abits} x {bbits} bits", flush=True)
    want = O.fft_mul(a, abits, b, bbits)
    got = eng.mul(a, abits, b, bbits)
    n = min(got.size, want.size)
    assert np.array_equal(got[:n], want[:n]) and not got[n:].any() and not want[n:].any()
    assert np.array_equal(eng.mul(b, bbits, a, abits), got)


@pytest.mark.parametrize("r,n,on", W.SLABS)
def test_slab(eng, r, n, on):
    from mersenne_trinomial_amd._capi import check, lib
    from mersenne_trinomial_amd.device import DeviceBuffer
    nw = O.words(r)
    pitch = nw + 5
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
        print(f"r={r} n={n} add_x={add_x}", flush=True)
        check(lib.gf2t_mulmod_slab(A.ptr, pitch, B.ptr, pitch, add_x, r, S.ptr, out.ptr, pitch, n, work.ptr, None))
        got = out.download().reshape(n, pitch)
        for i in (0, 1, n // 2, n - 1):
            t = b[i, :nw].copy()
            t[0] ^= np.uint64(2 * add_x)
            assert np.array_equal(got[i, :nw], O.mulmod(a[i, :nw].copy(), r, t, r, r, int(s[i]))), (add_x, i)
