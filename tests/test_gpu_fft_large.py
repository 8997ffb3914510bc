"""Transforms of 2^21 to 2^27 points, where the twiddles of the low levels (from
2^23 points on) and of a butterfly window (from 2^25) lie in GF(2^32): against
the oracle's transform, or its polynomial at single points, and back.
Bit-exact."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [21, 22, 23, 24, 25, 26, 27])
def test_transform(m):
    import mersenne_trinomial_amd as M
    from mersenne_trinomial_amd import device
    device.init(0)
    rng = np.random.default_rng(m)
    f = rng.integers(0, 2**64, 1 << m, dtype=np.uint64)
    print(f"2^{m} points", flush=True)
    F = M.fft_fwd(f, m)
    if m <= 23:
        assert np.array_equal(F, O.fft_fwd(f, m))
    basis = O.cantor_basis()
    for i in [0, (1 << m) - 1] + [int(x) for x in rng.integers(0, 1 << m, 4)]:
        assert int(F[i]) == O.poly_eval64(f, O.cantor_point(basis, i)), i
    assert np.array_equal(M.fft_fwd(F, m, inverse=True), f)
