"""Launches that take another tile of their instance (grids that leave the device idle) against the same launch on the instance's own
tile: equal bit for bit over grids on both sides of the rule, ragged M, N and K, batches, im2col and window convs, channels first
and expanded input; what an instance refuses, it refuses whatever tile the launch would take; capture with tiles that are
not loaded yet."""
import ctypes

import numpy as np
import pytest
import torch

from heron_amd import backend as B
from heron_amd import hostops, instances, tuned
from heron_amd.ops.rocm import getOpFromName

pytestmark = pytest.mark.gpu

D, F16, U8, GEMM, CONV = instances.D, instances.F16, instances.U8, instances.GEMM, instances.CONV
GEMMS = {
    "small": instances.BEST["small"], "small_f16": instances.BEST["small_f16"],
    "u8-128": D(U8, GEMM, 128, 128, 128, 2, 2, 16, 2, 1, epi=1, colsum=1, nt=1),
    "f16-128": D(F16, GEMM, 128, 128, 128, 2, 2, 32, 2, 1, nt=1),
    "f16-256": tuned.load("gemm_f16_8192").desc, "u8-256": tuned.load("gemm_u8s8_8192").desc, "pv": tuned.load("bmm_f16_pv").desc,
}
CONVS = {
    "f16-64": D(F16, CONV, 128, 64, 128, 2, 1, 32, 2, 1, epi=1), "f16-128": D(F16, CONV, *instances.PARITY_SHAPES[2]),
    "u8-64": D(U8, CONV, 128, 64, 128, 2, 2, 16, 3, 1, epi=1, colsum=1),
    "f16-window": tuned.load("conv2d_f16_resnet").desc, "u8-window": tuned.load("conv2d_u8s8_resnet").desc,
}


def _operands(f16, a, b, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if f16:
        return torch.randn(a, device="cuda", generator=gen).half(), torch.randn(b, device="cuda", generator=gen).half()
    return (torch.randint(0, 256, a, device="cuda", generator=gen, dtype=torch.uint8),
            torch.randint(-128, 128, b, device="cuda", generator=gen, dtype=torch.int8))


def _cut(mod, p):
    return mod.launch_tile(p).as_tuple() != mod.desc.as_tuple()


@pytest.mark.parametrize("name", sorted(GEMMS))
def test_gemm(name, hrn):
    d = GEMMS[name]
    mod, own, f16 = B.Module(d), B.Module(d, own_tiles=True), d.dtype == F16
    taken = set()
    for i, (b, m, n, k) in enumerate([(1, 64, 64, 64), (1, 1, 4, 16), (1, 65, 68, 1040), (1, 1111, 1500, 2064), (3, 130, 36, 304), (1, 2048, 1024, 256),
                                      (1, 1025, 2052, 128), (1, 2049, 580, 208), (40, 182, 64, 96), (1, 4100, 4100, 80)]):
        A, W = _operands(f16, (b, m, k), (b, n, k), i)
        if b == 1:
            A, W = A[0], W[0]
        if (n % 8 and f16) and d.epilogue:
            for x in (mod, own):
                with pytest.raises(B.HeronRocmError):
                    hostops.gemm(x, A, W)
            continue
        p = B.gemm_problem(b, m, n, k)
        assert not _cut(own, p)
        t = mod.launch_tile(p)
        taken.add((t.bm, t.bn, t.wm, t.wn))
        tiles = -(-m // d.bm) * -(-n // d.bn) * b
        few_waves = d.wm * d.wn < 4 and (256 < tiles <= 6 * 256 or (tiles <= 256 and k * (2 if f16 else 1) > 2 * d.bkb))
        assert _cut(mod, p) == (few_waves or (tiles <= 128 and (d.bm > 64 or d.bn > 64)))
        print("tiles gemm", name, (b, m, n, k), t.as_tuple(), flush=True)
        bsum = hostops.column_sums(W) if d.colsum else None
        assert torch.equal(hostops.gemm(mod, A, W, bsum=bsum), hostops.gemm(own, A, W, bsum=bsum))
    assert len(taken) >= 2
    mod.close()
    own.close()


@pytest.mark.parametrize("name", sorted(CONVS))
def test_conv(name, hrn):
    d = CONVS[name]
    mod, own, f16 = B.Module(d), B.Module(d, own_tiles=True), d.dtype == F16
    cases = [(1, 7, 9, 64, 64, 3, 1, 1, 1), (8, 28, 31, 64, 64, 5, 1, 2, 1), (3, 17, 16, 64, 80, 3, 1, 1, 1), (33, 56, 56, 64, 72, 1, 1, 0, 1), (20, 57, 55, 64, 64, 3, 1, 1, 1)]
    if not d.conv_window:
        cases += [(2, 15, 15, 80, 48, 3, 2, 1, 1), (1, 9, 9, 112, 16, 5, 1, 4, 2), (16, 27, 27, 128, 80, 3, 1, 1, 1)]
    cut = 0
    for i, (n, h, w, ci, co, k, s, pd, dl) in enumerate(cases):
        X, F = _operands(f16, (n, h, w, ci), (co, k, k, ci), i)
        cut += _cut(mod, B.conv2d_problem(n, h, w, ci, co, k, k, s, pd, dl))
        print("tiles conv", name, cases[i], flush=True)
        bsum = hostops.column_sums(F) if d.colsum else None
        assert torch.equal(hostops.conv2d_nhwc(mod, X, F, s, pd, dl, bsum=bsum), hostops.conv2d_nhwc(own, X, F, s, pd, dl, bsum=bsum))
    assert cut >= 2 and (cut < len(cases) or d.conv_window)
    mod.close()
    own.close()


@pytest.mark.parametrize("name", sorted(CONVS))
def test_channels_first(name, hrn):
    d = CONVS[name]
    mod, own, f16 = B.Module(d), B.Module(d, own_tiles=True), d.dtype == F16
    for op, args in [("c2d_nchw", [3, 13, 11, 64, 72, 3, 3, 1, 1, 1]), ("c1d", [2, 301, 64, 64, 3, 1, 1, 1]), ("t2d", [2, 9, 7, 64, 96, 1, 1, 2, 0, 1, 0]),
                     ("t2d", [16, 56, 56, 64, 128, 1, 1, 2, 0, 1, 0]), ("t2d", [2, 9, 7, 128, 40, 3, 3, 2, 1, 1, 1])]:
        ctx = type("Ctx", (), dict(set_info=lambda self, i: setattr(self, "info", i), set_axis_map=lambda self, m: None))()
        getOpFromName(op)(ctx, *args, *(["float16"] * 2 if f16 else ["int8"] * 2))
        info, c = ctx.info, ctx.info["conv"]
        if d.conv_window and (2 * c["pad"] != c["KH"] - 1 or 2 * c["pad_w"] != c["KW"] - 1):
            continue
        inputs = list(_operands(f16, info["reference_args"]["input"], info["reference_args"]["filter"], len(args)))
        print("tiles channels first", name, op, args, flush=True)
        assert torch.equal(hostops.run_operator(mod, info, inputs), hostops.run_operator(own, info, inputs))
    mod.close()
    own.close()


def test_refusals_are_the_instances_own(hrn):
    """A window too large for the instance's tile is refused although a smaller tile's window would fit."""
    d = CONVS["f16-window"]
    mod = B.Module(d)
    X, F = _operands(True, (1, 20, 200, 128), (64, 3, 3, 128), 1)
    with pytest.raises(B.HeronRocmError, match="exceeds 163840"):
        hostops.conv2d_nhwc(mod, X, F, 1, 1, 1)
    mod.close()


def test_first_launch_under_capture(hrn):
    d = GEMMS["u8-128"]
    mod, own = B.Module(d), B.Module(d, own_tiles=True)
    A, W = _operands(False, (300, 528), (260, 528), 3)
    bsum = hostops.column_sums(W)
    out = torch.empty((300, 260), dtype=torch.int32, device="cuda")
    hostops.gemm(own, A, W, bsum=bsum)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        hostops.gemm(mod, A, W, out=out, bsum=bsum)
    for _ in range(3):
        A.random_(0, 256)
        out.fill_(1)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, hostops.gemm(own, A, W, bsum=bsum))
    mod.close()
    own.close()
