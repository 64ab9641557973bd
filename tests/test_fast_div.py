"""The multipliers the kernels divide by: n / d as (2n * m >> 32) >> shift, for every n below 2^31."""
import random

import pytest


def fast_div(d):
    shift = (d - 1).bit_length()
    return ((1 << (31 + shift)) + d - 1) // d, shift


@pytest.mark.parametrize("d", [1, 2, 3, 5, 7, 8, 56, 58, 63, 64, 65, 892, 898, 3136, 12321, 65535, 65537, (1 << 30) - 1, 1 << 30, (1 << 30) + 1, (1 << 31) - 1])
def test_quotients(d):
    m, shift = fast_div(d)
    assert m < 1 << 32
    rng = random.Random(d)
    top = (1 << 31) - 1
    ns = {0, 1, d - 1, d, d + 1, top - 1, top, top // d * d - 1, top // d * d}
    for q in (1, 2, 3, top // d, top // d - 1):
        ns.update((q * d - 1, q * d, q * d + 1))
    ns.update(rng.randrange(top + 1) for _ in range(2000))
    for n in ns:
        if 0 <= n <= top:
            assert ((2 * n * m) >> 32) >> shift == n // d, n
