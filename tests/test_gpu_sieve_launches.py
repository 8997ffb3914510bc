"""The sieve at the edges of its launch rules, against the oracle: periods
that are and are not below smax, degree ranges that start above some of
their divisors, few and many s per thread of the sweep, and a prior image."""
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


# smax about 2^d - 1; 524288 values for each s per thread
@pytest.mark.parametrize("r,dmin,dmax,smax", [
    (4423, 2, 12, 2211), (9689, 2, 13, 4094), (9689, 2, 13, 4095), (9689, 2, 13, 4096),
    (5, 2, 3, 2), (3021377, 2, 20, 1048574), (3021377, 2, 20, 1048575), (3021377, 11, 21, 1510688),
    (3021377, 7, 16, 524288), (3021377, 20, 21, 524289), (3021377, 19, 23, 300000), (132049, 16, 17, 66024)])
def test_ranges(eng, r, dmin, dmax, smax):
    best, st = eng.run_gpu(r, dmax, smax, min_depth=dmin)
    want, _ = O.sieve(r, dmax, smax, dmin=dmin, nthreads=8)
    assert np.array_equal(best, want)
    assert [s.classes for s in st] == [O.count_irreducible(s.d) for s in st]


def test_prior_image_keeps_the_least(eng):
    """The sweep and the marks only lower a key."""
    r, smax = 132049, 66024
    rng = np.random.default_rng(5)
    prior = np.full(smax + 1, O.NONE, np.uint64)
    prior[rng.integers(1, smax + 1, 9000)] = np.uint64((2 << 48) | 7)
    prior[rng.integers(1, smax + 1, 9000)] = np.uint64((12 << 48) | 1)
    prior[rng.integers(1, smax + 1, 9000)] = np.uint64((19 << 48) | (1 << 20) - 1)
    got, _ = eng.run_gpu(r, 18, smax, best=prior.copy())
    want, _ = O.sieve(r, 18, smax, nthreads=8)
    assert np.array_equal(got, np.minimum(prior, want))


def test_r_not_prime_to_the_period_is_refused(eng):
    from mersenne_trinomial_amd._capi import GF2TError
    with pytest.raises(GF2TError, match="d=5"):
        eng.run_gpu(31, 5, 15)
    best, _ = eng.run_gpu(31, 4, 15)
    assert np.array_equal(best, O.sieve(31, 4, 15)[0])
