"""The sieve's class logarithms on the host: the functions its kernels call
(csrc/class_log.hpp) against the general ones and plain Python, exactly."""
import ctypes as C
import math
import os
import random
import subprocess

import numpy as np
import pytest

import oracle as O

HERE = os.path.dirname(os.path.abspath(__file__))
P32 = C.POINTER(C.c_uint32)


@pytest.fixture(scope="module")
def cl(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("cl") / "class_log.so")
    subprocess.run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-shared", "-fPIC", "-w", "-o", so,
                    os.path.join(HERE, "host", "class_log.cpp")], check=True)
    lib = C.CDLL(so)
    lib.cl_minpoly.restype = lib.cl_minpoly_bm.restype = C.c_uint64
    lib.cl_log.restype = C.c_uint32
    lib.cl_maps.argtypes = [C.c_uint64, C.c_int, P32]
    lib.cl_minpoly.argtypes = [C.c_uint32, C.c_int, P32]
    lib.cl_minpoly_bm.argtypes = [C.c_uint32, C.c_uint64, C.c_int, C.c_uint32]
    lib.cl_fill.argtypes = [P32, P32, C.c_uint64, C.c_int, P32, P32]
    lib.cl_log.argtypes = [C.c_uint64, C.c_int, P32, P32]
    lib.cl_progressions.argtypes = [P32, P32, C.c_int, P32, C.c_int, P32, P32]
    lib.cl_lyndon.argtypes = [C.c_uint32, C.c_int]
    lib.cl_prefix.argtypes = [C.c_uint32, C.c_int]
    lib.cl_is_lyndon32.argtypes = [C.c_uint32, C.c_int, C.c_uint32]
    return lib


def p32(a):
    return a.ctypes.data_as(P32)


def prim(d):
    from mersenne_trinomial_amd._capi import lib
    return int(lib.gf2t_primitive_poly(d))


def mul(a, b, q, d):
    t = 0
    for i in range(d):
        if (b >> i) & 1:
            t ^= a << i
    for i in range(2 * d - 2, d - 1, -1):
        if (t >> i) & 1:
            t ^= q << (i - d)
    return t


def clmul(a, b):
    t = 0
    while b:
        t ^= a * (b & -b)
        b &= b - 1
    return t


@pytest.mark.parametrize("d", list(range(2, 17)))
def test_lyndon_words_and_prefixes(cl, d):
    M = 2**d - 1
    lb = min(11, d - 1)
    found = 0
    for w in range(1 << (d - lb - 1)):
        viable = cl.cl_prefix(w, d - lb)
        for low in range(1, 1 << lb, 2):
            j = (w << lb) | low
            got = cl.cl_lyndon(j, d)
            assert got == cl.cl_is_lyndon32(j, d, M), j
            assert viable or not got, j
            found += got
    assert found == O.count_irreducible(d)


@pytest.mark.parametrize("d", [27, 30, 31, 32])
def test_lyndon_words_large(cl, d):
    rng = random.Random(d)
    M = 2**d - 1
    for _ in range(20000):
        j = rng.getrandbits(d - 1 - rng.randint(0, 8)) | 1
        if rng.random() < .3:      # words that repeat, or nearly
            h = rng.choice([k for k in range(1, d) if d % k == 0])
            b = j & (2**h - 1)
            j = sum(b << (h * i) for i in range(d // h)) ^ (rng.random() < .5)
        ok = cl.cl_lyndon(j, d)
        if j & 1 and not j >> (d - 1):
            assert ok == cl.cl_is_lyndon32(j, d, M), j
        assert not ok or all(cl.cl_prefix(j >> (d - n), n) for n in range(1, d))


@pytest.mark.parametrize("d", list(range(2, 15)))
def test_class_logarithms(cl, d):
    q, M = prim(d), 2**d - 1
    m = np.zeros(4096, np.uint32)
    assert cl.cl_maps(q, d, p32(m))
    g = [1]
    for _ in range(M - 1):
        g.append(mul(g[-1], 2, q, d))
    js = np.array([j for j in range(1, M) if cl.cl_is_lyndon32(j, d, M)], np.uint32)
    T = np.zeros(1 << (d - 2), np.uint32)
    cl.cl_fill(p32(js), p32(np.array([g[j] for j in js], np.uint32)), len(js), d, p32(m), p32(T))
    assert np.count_nonzero(T) == len(js)      # one slot for each class
    for j in js.tolist():
        for i in range(d):
            e = (j << i) % M
            assert cl.cl_log(g[e], d, p32(m), p32(T)) == e
            a = random.Random(e).randrange(M)  # as an unreduced product
            assert cl.cl_log(clmul(g[a], g[(e - a) % M]), d, p32(m), p32(T)) == e


@pytest.mark.parametrize("d", [2, 3, 8, 12, 16, 20, 21, 24, 30, 31, 32])
def test_minimal_polynomials(cl, d):
    q = prim(d)
    m = np.zeros(4096, np.uint32)
    assert cl.cl_maps(q, d, p32(m))
    tmask = 0
    for i in range(d):
        y = t = 1 << i if i < d else 0
        for _ in range(d - 1):
            y = mul(y, y, q, d)
            t ^= y
        tmask |= t << i
    rng = random.Random(d)
    n = 0
    for _ in range(60):
        beta = rng.randrange(2, 2**d)
        want = cl.cl_minpoly_bm(beta, q, d, tmask)
        assert cl.cl_minpoly(beta, d, p32(m)) == want
        n += want != 0
    assert n


@pytest.mark.parametrize("d", [2, 3, 4, 6, 9, 12, 18, 20, 21, 24, 30, 31, 32])
def test_progressions(cl, d):
    """Every kind of gcd(j, 2^d - 1), square factors (6, 12, 18, 20, 21, 24,
    30) among them."""
    M = 2**d - 1
    ps = [p for p in range(3, 70000) if M % p == 0 and all(p % k for k in range(2, math.isqrt(p) + 1))]
    left = M
    for p in ps:
        while left % p == 0:
            left //= p
    if left > 1:
        ps.append(left)
    primes = np.array(ps, np.uint32)
    rng = random.Random(d)
    divs = [k for k in range(1, 5000) if M % k == 0] + ps
    j, v = [], []
    for _ in range(4096):
        g = rng.choice(divs)
        x = rng.randrange(1, max(2, M // g + 1)) * g % M or 1
        if x < M:
            j.append(x)
            v.append(rng.randrange(M) // g * g if rng.random() < .8 else rng.randrange(M))
    k = len(j) // 8 * 8
    j, v = np.array(j[:k], np.uint32), np.array(v[:k], np.uint32)
    n, s = np.zeros_like(j), np.zeros_like(j)
    for c0 in range(0, k, 8):
        cl.cl_progressions(p32(j[c0:]), p32(v[c0:]), d, p32(primes), len(primes), p32(n[c0:]), p32(s[c0:]))
    for a, b, nn, ss in zip(j.tolist(), v.tolist(), n.tolist(), s.tolist()):
        g = math.gcd(a, M)
        if b % g:
            assert nn == 0
        else:
            assert nn == M // g and ss == b // g * pow(a // g, -1, nn) % nn, (a, b)
