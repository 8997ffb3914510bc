"""The rules by which products are launched, on the host.  No GPU."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

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
