"""Addresses of im2col loads: rows and taps that kernels carry from load to load against the definition, by the code that kernels run.
Filters of unequal strides, pads and dilations, channels below and above a k-tile, K slices that begin inside a filter row, results
of fewer pixels than a load covers, zero-expanded inputs; and strides, pads and dilations at the ends of their range."""
import ctypes
import random

import pytest

from launch_args import library


def errors(n, h, w, ci, kh, kw, sy, sx, py, px, dy, dx, es, row_bytes, rows, loads, expanded=(0, 0)):
    ho = (h + 2 * py - (kh - 1) * dy - 1) // sy + 1
    wo = (w + 2 * px - (kw - 1) * dx - 1) // sx + 1
    assert ho > 0 and wo > 0
    conv = (ctypes.c_int * 16)(n, h, w, ci, ho, wo, kh, kw, sy, py, dy, sx, px, dx, *expanded)
    kts = -(-kh * kw * ci * es // row_bytes)
    starts = sorted({0, min(1, kts - 1), kts // 3, kts // 2})
    f = library().conv_walk_errors
    f.restype = ctypes.c_longlong
    return f(conv, es, row_bytes, rows, loads, (ctypes.c_int * len(starts))(*starts), len(starts))


@pytest.mark.parametrize("seed", range(60))
def test_random_convs(seed):
    rng = random.Random(seed)
    es = rng.choice([1, 2])
    row_bytes = rng.choice([64, 128, 256])
    while True:
        kh, kw = rng.choice([1, 2, 3, 5, 7]), rng.choice([1, 2, 3, 5])
        h, w = rng.randint(1, 40), rng.randint(1, 70)
        sy, sx, dy, dx = (rng.randint(1, 3) for _ in range(4))
        py, px = rng.randint(0, kh * dy), rng.randint(0, kw * dx)
        if h + 2 * py > (kh - 1) * dy and w + 2 * px > (kw - 1) * dx:
            break
    ci = rng.choice([16, 32, 48, 80, 112, 144, 176, 208, 272])
    rows = rng.choice([4, 8, 16, 32, 64])
    assert errors(rng.randint(1, 9), h, w, ci, kh, kw, sy, sx, py, px, dy, dx, es, row_bytes, rows, rng.choice([1, 2, 4])) == 0
    if sy == sx == 1:
        assert errors(3, h, w, ci, kh, kw, 1, 1, py, px, dy, dx, es, row_bytes, rows, 4, expanded=((h + 1) // 2, (w + 1) // 2)) == 0


G = 1 << 30


@pytest.mark.parametrize("conv", [
    # n, h, w, ci, kh, kw, stride, pad, dilation as (height, width) pairs
    (2, 9, 9, 64, 1, 1, (1 << 26, 1 << 26), (0, 0), (1, 1)),                 # one pixel of each image
    (3, 5, 7, 64, 3, 3, (G, 2 * G - 1), (1, 1), (1, 1)),
    (1, 1, 3 << 22, 16, 1, 1, (1, 1 << 23), (0, 0), (1, 1)),                 # a step of 2^28 input pixels
    (2, 1, 1, 64, 1, 1, (G, G), (G, G), (1, 1)),                             # three rows of three: the extent of the result is 3 * 2^30
    (2, 3, 3, 48, 2, 2, (1, 1), (G // 2, G // 2), (G, G)),                   # the extent of the taps is 2^31
    (1, 4, 4, 128, 3, 3, (G // 2, G // 2), (G // 2, G // 2), (G // 2, G // 2)),
    (1, 3, 3, 32, 5, 5, (1, 1), (2 * G - 1, 2 * G - 1), (G, G)),             # taps a multiple of 2^32 apart
    (4, 6, 6, 32, 1, 1, (2, 2), (0, 0), (G, 2 * G - 1)),                     # dilation of a single tap
])
@pytest.mark.parametrize("es,row_bytes", [(2, 128), (1, 64), (2, 64)])
def test_far_strides_pads_and_dilations(conv, es, row_bytes):
    n, h, w, ci, kh, kw, s, p, d = conv
    assert errors(n, h, w, ci, kh, kw, *s, *p, *d, es, row_bytes, 32, 4) == 0
