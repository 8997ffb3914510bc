"""A product's workspace serves every product of no larger operands: the
bytes grow with either operand, across the rule that picks how small
products are formed."""
import random

from mersenne_trinomial_amd._capi import lib


def test_mul_workspace_grows_with_either_operand():
    w = lambda ca, cb: lib.gf2t_mul_workspace_bytes(32 * ca, 32 * cb)
    edges = [1, 2, 127, 128, 129, 511, 512, 513, 1022, 1023, 1024, 1025, 2047, 2048, 4127, 8191, 8192,
             10239, 10240, 10241, 16384, 32768, 65535, 65536, 65537, 200000]
    for ca in edges:
        for a, b in zip(edges, edges[1:]):
            assert w(ca, a) <= w(ca, b), (ca, a, b)
            assert w(a, ca) <= w(b, ca) and w(a, ca) == w(ca, a), (ca, a, b)
    rng = random.Random(1)
    for _ in range(20000):
        ca, cb = (int(2 ** rng.uniform(0, 18)) for _ in range(2))
        assert w(ca, cb) <= w(ca + rng.randint(0, 3), cb + rng.randint(0, 3)), (ca, cb)
