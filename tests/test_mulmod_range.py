"""Moduli past the folds' limit are refused whatever the operands' size,
before anything is launched.  No GPU: the buffers are never read."""
import ctypes as C

import pytest

from mersenne_trinomial_amd._capi import lib

EINVAL = -1


@pytest.mark.parametrize("bits", [1, 1000, 16384])
def test_small_product_of_a_large_modulus(bits):
    buf = (C.c_uint64 * 1024)()
    p = C.addressof(buf)
    for r in (1 << 34, (1 << 34) + 5, 1 << 40):
        assert lib.gf2t_mulmod(p, bits, p, bits, r, 7, p, p, None) == EINVAL
        assert b"2^34" in lib.gf2t_last_error()
