"""Squaring chains at the edges of their launch rules, against the oracle:
chains held in LDS (the residue that just fits and the one that does not,
one and several pairs per thread, chains longer than one launch), units
shortened for launches of few tiles, and batches whose chains differ in
length (an odd one takes its single squaring in the first launch).
Bit-exact."""
import ctypes as C

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
LDS_BITS = 64 * 10238   # the largest residue that runs in LDS


@pytest.fixture(scope="module")
def eng():
    import mersenne_trinomial_amd as M
    from mersenne_trinomial_amd import device
    device.init(0)
    return M


def rand_res(rng, r):
    a = rng.integers(0, 2**64, O.words(r), dtype=np.uint64)
    if r & 63:
        a[-1] &= np.uint64((1 << (r & 63)) - 1)
    return a


# 3 steps and more run in LDS up to LDS_BITS; 2048 pairs take two per thread
@pytest.mark.parametrize("r", [3, 5, 64, 127, 128, 129, 8192, 131072, 131073, 262143, 262144,
                               393217, LDS_BITS - 1, LDS_BITS, LDS_BITS + 1])
def test_chain_edges(eng, r):
    rng = np.random.default_rng(r)
    for s in sorted({1, 2, r // 3, (r - 1) // 2} & set(range(1, (r + 1) // 2))):
        a = rand_res(rng, r)
        for k in (0, 3, 4):
            assert np.array_equal(eng.square_fold(a, r, s, k), O.square_fold_steps(a, r, s, k)), (s, k)


@pytest.mark.parametrize("k", [4095, 4096, 4097, 8193])
def test_chain_longer_than_a_launch(eng, k):
    x = rand_res(np.random.default_rng(k), 521)
    assert np.array_equal(eng.square_fold(x, 521, 48, k), O.square_fold_steps(x, 521, 48, k))


# (r, s, steps): in LDS and by launches, odd and even, equal and 64-fold r
BATCHES = [
    [(LDS_BITS, 1000, 5), (LDS_BITS + 1, 1000, 5), (LDS_BITS + 64, 3, 4), (521, 32, 1)],
    [(756839, 1, 1), (756839, 378419, 2), (756839, 3000, 3), (700032, 350015, 0)],
    [(3021377, 1510688, 7), (859433, 288477, 6), (132049, 2, 9), (44497, 22248, 5000)],
    [(859433, 7, 2), (859433, 429716, 2)],
    [(6972593, 3486296, 4), (65536 * 16, 65535, 3), (65536 * 16 + 64, 65537, 5), (859433, 1, 7)],
    [(37156667, 18578333, 4), (859433, 3, 2)],
    [(37156667, 5, 3), (43112609, 9000000, 5), (3021377, 77, 1)],
]


@pytest.mark.parametrize("cases", BATCHES, ids=["edge", "odd", "mixed", "even", "ranges", "columns", "columns-odd"])
def test_batch_edges(eng, cases):
    from mersenne_trinomial_amd._capi import check, lib
    from mersenne_trinomial_amd.device import DeviceBuffer
    rng = np.random.default_rng(len(cases))
    ins = [rand_res(rng, r) for r, _, _ in cases]
    bufs = [DeviceBuffer.from_array(a) for a in ins]
    tmps = [DeviceBuffer.words(O.words(r)) for r, _, _ in cases]
    n = len(cases)
    P = C.POINTER(C.c_uint64)
    rr, ss, kk = (np.array([c[j] for c in cases], dtype=np.uint64) for j in range(3))
    check(lib.gf2t_square_fold_batch((C.c_void_p * n)(*[b.ptr for b in bufs]),
                                     (C.c_void_p * n)(*[t.ptr for t in tmps]),
                                     rr.ctypes.data_as(P), ss.ctypes.data_as(P),
                                     kk.ctypes.data_as(P), n, None))
    for (r, s, k), a, b in zip(cases, ins, bufs):
        assert np.array_equal(b.download(O.words(r)), O.square_fold_steps(a, r, s, k)), (r, s, k)


@pytest.mark.parametrize("s", [1, 8, 65536, 11000000, 18578333])
@pytest.mark.parametrize("k", [1, 2, 4])
def test_windows_in_columns(eng, s, k):
    r = 37156667   # more than an XCD's L2: ranges in columns s apart
    a = rand_res(np.random.default_rng(s), r)
    assert np.array_equal(eng.square_fold(a, r, s, k), O.square_fold_steps(a, r, s, k))


def test_two_squaring_launches_above_the_windows_bound(eng):
    """A batch of more ranges than F^8 windows are used for: two squarings
    per launch, one in the first for the odd chain."""
    from mersenne_trinomial_amd._capi import check, lib
    from mersenne_trinomial_amd.device import DeviceBuffer
    r, n = 136279841, 9
    rng = np.random.default_rng(9)
    svals = [474, 1, 68139920, 40000001, 3, 65536, 30000000, 1000003, 9]
    steps = [4, 3, 2, 1, 4, 5, 3, 0, 2]
    ins = [rand_res(rng, r) for _ in range(n)]
    bufs = [DeviceBuffer.from_array(a) for a in ins]
    tmps = [DeviceBuffer.words(O.words(r)) for _ in range(n)]
    P = C.POINTER(C.c_uint64)
    rr, ss, kk = (np.array(v, dtype=np.uint64) for v in ([r] * n, svals, steps))
    check(lib.gf2t_square_fold_batch((C.c_void_p * n)(*[b.ptr for b in bufs]),
                                     (C.c_void_p * n)(*[t.ptr for t in tmps]),
                                     rr.ctypes.data_as(P), ss.ctypes.data_as(P),
                                     kk.ctypes.data_as(P), n, None))
    for s, k, a, b in zip(svals, steps, ins, bufs):
        assert np.array_equal(b.download(O.words(r)), O.square_fold_steps(a, r, s, k)), (s, k)
