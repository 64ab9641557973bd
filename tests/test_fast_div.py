"""The multipliers the kernels divide by: n / d for every n below 2^31, by the code that launches and kernels share."""
import ctypes
import random

import numpy as np
import pytest

from launch_args import library

_P = ctypes.POINTER(ctypes.c_uint32)


@pytest.mark.parametrize("d", [1, 2, 3, 5, 7, 8, 56, 58, 63, 64, 65, 892, 898, 3136, 12321, 65535, 65537, (1 << 30) - 1, 1 << 30, (1 << 30) + 1, (1 << 31) - 1])
def test_quotients(d):
    rng = random.Random(d)
    top = (1 << 31) - 1
    ns = {0, 1, d - 1, d, d + 1, top - 1, top, top // d * d - 1, top // d * d}
    for q in (1, 2, 3, top // d, top // d - 1):
        ns.update((q * d - 1, q * d, q * d + 1))
    ns.update(rng.randrange(top + 1) for _ in range(2000))
    n = np.array(sorted(n for n in ns if 0 <= n <= top), dtype=np.uint32)
    out = np.empty_like(n)
    library().div_all(n.ctypes.data_as(_P), out.ctypes.data_as(_P), len(n), d)
    assert np.array_equal(out, n // np.uint32(d))
