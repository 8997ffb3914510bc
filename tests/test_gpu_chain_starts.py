"""Batches by what their chains' first launch takes and by how many squarings
a launch does near the bound of the windows, against the oracle: one squaring
first of residues in columns (r a multiple of 64 among them), a short chain by
two squarings a launch, a longer one by three.  Bit-exact."""
import ctypes as C

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
R = 136279841


@pytest.mark.parametrize("rs,k,check", [((37156667, 37156667), 1, (0, 1)), ((37156667, 37156672), 4, (0, 1)),
                                        ((R,) * 7, 3, (0, 6)), ((R,) * 7, 5, (1,)), ((R,) * 7, 1, (3,))])
def test_uniform_batch(rs, k, check):
    from mersenne_trinomial_amd import device
    from mersenne_trinomial_amd._capi import check as ok, lib
    from mersenne_trinomial_amd.device import DeviceBuffer
    device.init(0)
    rng = np.random.default_rng(k + len(rs))
    ins = []
    for r in rs:
        a = rng.integers(0, 2**64, O.words(r), dtype=np.uint64)
        if r & 63:
            a[-1] &= np.uint64((1 << (r & 63)) - 1)
        ins.append(a)
    svals = [int(rng.integers(1, (r + 1) // 2)) for r in rs]
    bufs, tmps = [DeviceBuffer.from_array(a) for a in ins], [DeviceBuffer.words(a.size) for a in ins]
    n, P = len(rs), C.POINTER(C.c_uint64)
    rr, ss, kk = (np.array(v, dtype=np.uint64) for v in (rs, svals, [k] * n))
    ok(lib.gf2t_square_fold_batch((C.c_void_p * n)(*[b.ptr for b in bufs]), (C.c_void_p * n)(*[t.ptr for t in tmps]),
                                  rr.ctypes.data_as(P), ss.ctypes.data_as(P), kk.ctypes.data_as(P), n, None))
    for i in check:
        assert np.array_equal(bufs[i].download(), O.square_fold_steps(ins[i], rs[i], svals[i], k)), i
