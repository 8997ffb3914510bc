"""The rules by which products are launched, on the host.  No GPU."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import wrapped_shapes as W

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "mersenne_trinomial_amd", "csrc")


@pytest.fixture(scope="module")
def pr(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("pr") / "libpr.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I" + CSRC, "-o", out,
                           os.path.join(HERE, "host", "product_rules.cpp")])
    return C.CDLL(out)


@pytest.mark.parametrize("n", [1, 5, 32767, 32768, 65534, 65535, 100001])
@pytest.mark.parametrize("sizes", [[9], [9, 0, 12]])
def test_groups_fit_a_grid(pr, n, sizes):
    """Every pair is in one group of its size, and a group's transforms, two
    a pair, fit the 65535 rows of a launch."""
    most = pr.pr_max_pairs()
    assert 2 * most <= 65535
    m = np.array([sizes[j % len(sizes)] for j in range(n)], np.int32)
    group, place, size = (np.zeros(max(n, 16), np.int32) for _ in range(3))
    p = lambda a: a.ctypes.data_as(C.POINTER(C.c_int))
    count = pr.pr_groups(p(m), n, p(group), p(place), p(size))
    group, place = group[:n], place[:n]
    assert np.array_equal(group >= 0, m > 0)
    for g in range(count):
        mine = np.flatnonzero(group == g)
        assert 1 <= mine.size <= most and np.all(m[mine] == size[g])
        assert np.array_equal(place[mine], np.arange(mine.size))


def size_of(ca, cb):
    m = 1
    while (1 << m) < ca + cb - 1:
        m += 1
    return m if ca and cb else 0


def test_direct_pairs(pr):
    """Whole sizes from the smallest on, as long as their chunk pairs together
    are within the limit."""
    most = C.c_uint64(0)
    pr.pr_direct_pairs.restype = C.c_uint64
    most = pr.pr_direct_pairs()
    rng = np.random.default_rng(1)
    for _ in range(200):
        n, hi = int(rng.integers(1, 200)), rng.uniform(2, 18)
        ca, cb = (np.floor(2 ** rng.uniform(0, hi, n)).astype(np.uint64) for _ in range(2))
        ca[rng.random(n) < 0.1] = 0
        m = np.array([size_of(int(a), int(b)) for a, b in zip(ca, cb)], np.int32)
        v = np.zeros(n, np.int8)
        pr.pr_direct(m.ctypes.data_as(C.c_void_p), ca.ctypes.data_as(C.c_void_p),
                     cb.ctypes.data_as(C.c_void_p), n, v.ctypes.data_as(C.c_void_p))
        work = (ca * cb).astype(object)
        assert work[v == 1].sum() <= most and np.all(m[v == 1] > 0) and np.all(m[v == 1] <= 15)
        rest = m[(v == 0) & (m > 0)]
        if rest.size and rest.min() <= 15:   # the next size would pass the limit
            assert np.all(m[v == 1] < rest.min())
            assert work[v == 1].sum() + work[m == rest.min()].sum() > most


def test_batch_workspace_grows():
    """A batch's workspace serves every batch of fewer or shorter pairs."""
    from mersenne_trinomial_amd._capi import lib
    rng = np.random.default_rng(2)
    U = lambda v: (C.c_uint64 * len(v))(*[int(x) for x in v])
    size = lambda a, b: lib.gf2t_mulmod_batch_workspace_bytes(len(a), U(a), U(b))
    for _ in range(300):
        n, hi = int(rng.integers(1, 60)), rng.uniform(3, 23)
        a, b = (np.floor(2 ** rng.uniform(0, hi, n)) for _ in range(2))
        keep = rng.random(n) < 0.7
        keep[0] = True
        fa, fb = (np.floor(v * np.where(rng.random(n) < 0.5, 1, rng.random(n))) for v in (a, b))
        assert size(fa[keep], fb[keep]) <= size(a, b)


def wrap(pr, ca, cb, n):
    mp, ms, e = C.c_int(), C.c_int(), C.c_uint64()
    pr.pr_wrap.argtypes = [C.c_uint64] * 3 + [C.c_void_p] * 3
    on = pr.pr_wrap(ca, cb, n, C.addressof(mp), C.addressof(ms), C.addressof(e))
    return bool(on), mp.value, ms.value, e.value


@pytest.mark.parametrize("mp,e,ca,on", W.PRODUCTS)
def test_wrapped_products(pr, mp, e, ca, on):
    """The shapes that the GPU tests run lie where they are meant to."""
    got = wrap(pr, ca, W.other(mp, e, ca), 1)
    assert got[0] == on
    if on:   # the transforms fit those of an ordinary product
        assert got[1] == mp and got[3] == e and 2 * e - 1 <= 1 << got[2] and got[2] < mp


@pytest.mark.parametrize("r,n,on", W.SLABS)
def test_wrapped_slabs(pr, r, n, on):
    assert wrap(pr, W.chunks(r), W.chunks(r), n)[0] == on
