"""Launches that take another tile of their instance (grids that leave the device idle) against the same launch on the instance's own
tile: equal bit for bit over grids on both sides of the rule, ragged M, N and K, batches, im2col and window convs, channels first
and expanded input; what an instance refuses, it refuses whatever tile the launch would take; capture with tiles that are
not loaded yet."""
import os
import shutil

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


def _declared(op, args, f16):
    """(info, inputs) of an operator"""
    ctx = type("Ctx", (), dict(set_info=lambda self, i: setattr(self, "info", i), set_axis_map=lambda self, m: None))()
    getOpFromName(op)(ctx, *args, *(["float16"] * 2 if f16 else ["int8"] * 2))
    ref = ctx.info["reference_args"]
    return ctx.info, list(_operands(f16, ref["input"], ref["filter"], len(args)))


def _cut(mod, p, **how):
    return mod.launch_tile(p, **how).as_tuple() != mod.desc.as_tuple()


def _conv_problem(info):
    c = info["conv"]
    return B.conv2d_problem(*(c[n] for n in ("N", "H", "W", "CI", "CO", "KH", "KW")), (c["stride"], c["stride_w"]), (c["pad"], c["pad_w"]),
                            (c["dil"], c["dil_w"]))


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
    cut = 0
    for op, args in [("c2d_nchw", [3, 13, 11, 64, 72, 3, 3, 1, 1, 1]), ("c1d", [2, 301, 64, 64, 3, 1, 1, 1]), ("t2d", [2, 9, 7, 64, 96, 1, 1, 2, 0, 1, 0]),
                     ("t2d", [16, 56, 56, 64, 128, 1, 1, 2, 0, 1, 0]), ("t2d", [2, 9, 7, 128, 40, 3, 3, 2, 1, 1, 1])]:
        info, inputs = _declared(op, args, f16)
        c = info["conv"]
        if d.conv_window and (2 * c["pad"] != c["KH"] - 1 or 2 * c["pad_w"] != c["KW"] - 1):
            continue
        p, expand = _conv_problem(info), op == "t2d" and args[7] > 1
        took = _cut(mod, p, chw=True, expand=expand)
        cut += took
        print("tiles channels first", name, op, args, mod.launch_tile(p, chw=True, expand=expand).as_tuple(), flush=True)
        assert not _cut(own, p, chw=True, expand=expand)
        assert torch.equal(hostops.run_operator(mod, info, inputs), hostops.run_operator(own, info, inputs))
        assert _cut(mod, p, chw=True, expand=expand) == took             # (also after its kernels were loaded)
    assert cut >= 3
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
    p = B.gemm_problem(1, 300, 260, 528)
    assert _cut(mod, p)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        hostops.gemm(mod, A, W, out=out, bsum=bsum)
    assert _cut(mod, p)                                                  # the tile was loaded inside the capture, else it is passed by
    for _ in range(3):
        A.random_(0, 256)
        out.fill_(1)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, hostops.gemm(own, A, W, bsum=bsum))
    mod.close()
    own.close()


def _copy_parts(tmp, *parts):
    """A cache that holds these (descriptor, kernels) and nothing else; kernels: "main", "chw" or "expand"."""
    for d, part in parts:
        stem = B.compile_desc(d)[:-len(".hsaco")]
        for end in (".hsaco", ".info") if part == "main" else ("_%s.hsaco" % part,):
            shutil.copy(stem + end, tmp)


@pytest.fixture
def no_compiler(tmp_path, monkeypatch):
    """An empty cache, and a compiler that only leaves a mark."""
    cache, script, mark = tmp_path / "cache", tmp_path / "hipcc", tmp_path / "called"
    cache.mkdir()
    script.write_text("#!/bin/sh\ntouch %s\nexit 1\n" % mark)
    script.chmod(0o755)

    def use():
        monkeypatch.setenv("HRN_CACHE_DIR", str(cache))
        monkeypatch.setenv("HRN_HIPCC", str(script))
    return cache, use, mark


def test_a_launch_compiles_no_tile(no_compiler, hrn):
    """An instance whose tiles are not in the cache launches its own, and neither the launch nor the questions about it compile."""
    cache, use, mark = no_compiler
    d = GEMMS["u8-128"]
    _copy_parts(cache, (d, "main"))
    A, W = _operands(False, (300, 528), (260, 528), 3)
    bsum, p = hostops.column_sums(W), B.gemm_problem(1, 300, 260, 528)
    own = B.Module(d, own_tiles=True)
    want = hostops.gemm(own, A, W, bsum=bsum)
    use()
    mod = B.Module(d)
    assert not _cut(mod, p) and mod.is_deep(p) == own.is_deep(p)
    assert torch.equal(hostops.gemm(mod, A, W, bsum=bsum), want)
    assert not mark.exists()
    mod.close()
    own.close()


def test_channels_first_without_the_tiles_kernels(no_compiler, hrn):
    """A channels-first launch whose tile lies in the cache without channels-first kernels takes the instance's own."""
    cache, use, mark = no_compiler
    d = CONVS["f16-128"]
    info, inputs = _declared("c2d_nchw", [2, 5, 6, 64, 8, 3, 3, 1, 1, 1], True)
    own = B.Module(d, own_tiles=True)
    want = hostops.run_operator(own, info, inputs)
    _copy_parts(cache, (d, "main"), (d, "chw"), *((t, "main") for t in B.tiles(d)))
    use()
    mod = B.Module(d)
    p = _conv_problem(info)
    assert _cut(mod, p) and not _cut(mod, p, chw=True)
    assert torch.equal(hostops.run_operator(mod, info, inputs), want)
    assert not mark.exists()
    mod.close()
    own.close()


def test_a_tile_that_cannot_be_loaded(no_compiler, hrn):
    """A code object without the kernel it should hold leaves the launch to the instance, and no error behind."""
    cache, use, mark = no_compiler
    d = CONVS["f16-128"]
    p = B.conv2d_problem(2, 5, 6, 64, 8, 3, 3, 1, 1, 1)
    X, F = _operands(True, (2, 5, 6, 64), (8, 3, 3, 64), 1)
    own = B.Module(d, own_tiles=True)
    want = hostops.conv2d_nhwc(own, X, F, 1, 1, 1)
    _copy_parts(cache, (d, "main"), *((t, "main") for t in B.tiles(d)))
    for t in B.tiles(d):
        stem = os.path.basename(B.compile_desc(t))[:-len(".hsaco")]
        shutil.copy(B.compile_desc(d)[:-len(".hsaco")] + "_chw.hsaco", cache / (stem + ".hsaco"))
    use()
    mod = B.Module(d)
    assert _cut(mod, p)
    for _ in range(2):
        assert torch.equal(hostops.conv2d_nhwc(mod, X, F, 1, 1, 1), want)
        assert not _cut(mod, p)
    assert "hipModule" not in B.lib().hrn_last_error().decode()
    torch.zeros(4, device="cuda").add_(1)
    torch.cuda.synchronize()
    mod.close()
    own.close()


# a window tile that has a CU to itself, on more tiles than half the CUs: (image width, channels, filter, whether two of the half fit a
# CU).  The 512x64 record's half: 32 KiB of stages, and 256 + 2 pad (width + 1) rows of 2 ci bytes in 48 KiB at width 63 (3x3) and 31 (5x5).
@pytest.mark.parametrize("w,ci,k,two", [(56, 64, 3, True), (60, 64, 3, True), (63, 64, 3, True), (64, 64, 3, False), (160, 64, 3, False),
                                        (31, 64, 5, True), (32, 64, 5, False), (80, 64, 5, False), (111, 64, 1, True), (57, 128, 1, False)])
def test_half_a_window_where_two_fit(w, ci, k, two, hrn):
    d = CONVS["f16-window"]
    mod, own = B.Module(d), B.Module(d, own_tiles=True)
    n = -(-200 * d.bm // (w * w))
    p = B.conv2d_problem(n, w, w, ci, 64, k, k, 1, k // 2, 1)
    t = mod.launch_tile(p)
    half = d.bm // 2 + 2 * (k // 2) * (w + 1)
    lds = t.stages * t.bn * t.bkb + -(-half * ci * 2 // 1024) * 1024
    assert two == (lds <= 80 * 1024)
    assert (t.bm, t.bn) == ((d.bm // 2 if two else d.bm), d.bn)
    X, F = _operands(True, (n, w, w, ci), (64, k, k, ci), w)
    print("half a window", w, ci, k, t.as_tuple(), flush=True)
    assert torch.equal(hostops.conv2d_nhwc(mod, X, F, 1, k // 2, 1), hostops.conv2d_nhwc(own, X, F, 1, k // 2, 1))
    mod.close()
    own.close()


def test_half_a_window_in_rows_only(hrn, tmp_path, monkeypatch):
    """A window tile wider than high is halved in columns where the grid leaves CUs idle, and never to share a CU."""
    monkeypatch.setenv("HRN_CACHE_DIR", str(tmp_path))
    d = D(F16, CONV, 64, 128, 256, 2, 4, 32, 2, 1, epi=1, win=1)
    for t in [d, B.tiles(d)[0]]:
        B.compile_desc(t)
    mod = B.Module(d)
    for n, tile in ((8, (64, 64)), (16, (64, 128))):                      # 98 and 196 tiles; 96 KiB of LDS, 64 KiB with half the columns
        t = mod.launch_tile(B.conv2d_problem(n, 28, 28, 256, 128, 1, 1, 1, 0, 1))
        assert (t.bm, t.bn) == tile
    mod.close()


@pytest.mark.parametrize("name", sorted(tuned.CASES))
def test_a_record_runs_its_own_tile_on_its_own_problem(name, hrn):
    t = tuned.load(name)
    _, op, shape, dtype = tuned.CASES[name]
    sched, _ = tuned.instantiate(name, op, shape, dtype, t.records)
    mod = B.Module(t.desc)
    assert not _cut(mod, sched.to_problem())
    mod.close()


def test_a_record_of_few_tiles(hrn):
    """On its own sizes, in any raster order, it keeps its tile; elsewhere the rule decides."""
    d = D(F16, GEMM, 256, 256, 128, 2, 4, 16, 2, 2)
    d.tuned_for = (1, 700, 520, 256)
    mod = B.Module(d)
    assert not _cut(mod, B.gemm_problem(1, 700, 520, 256, group_m=2))
    for other in (B.gemm_problem(1, 700, 520, 264), B.gemm_problem(1, 701, 520, 256), B.gemm_problem(1, 700, 528, 256), B.gemm_problem(2, 700, 520, 256)):
        assert _cut(mod, other)
    mod.close()
    d = CONVS["f16-128"]
    args = [2, 14, 14, 64, 48, 3, 3, 1, 1, 1]
    d.tuned_for = tuple(args)
    mod = B.Module(d)
    assert not _cut(mod, B.conv2d_problem(*args))
    for i, v in [(0, 3), (4, 64), (5, 5), (6, 1), (7, (1, 2)), (8, 2), (9, 2)]:
        assert _cut(mod, B.conv2d_problem(*args[:i], v, *args[i + 1:])), (i, v)
    assert _cut(mod, B.conv2d_problem(1, 28, 14, *args[3:]))             # as many pixels in another image
    mod.close()
