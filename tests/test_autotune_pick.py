"""The autotuner leaves a knob alone unless another value is clearly faster."""
import pytest


@pytest.mark.parametrize("times,default,want", [({9: 1.0, 11: 0.999, 13: 1.0}, 13, 13), ({9: 0.9, 11: 1.0}, 11, 9),
                                                ({9: 0.971, 11: 1.0}, 11, 11), ({9: 2.0, 10: 1.9}, 13, 10)])
def test_pick(times, default, want):
    from mersenne_trinomial_amd import autotune
    assert autotune.pick(times, default) == want
