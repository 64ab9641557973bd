"""Channels-first results stored by the conv kernels themselves, and zero-expanded inputs that are not in memory, against the
same instance with the layout passes around it (same products in the same order: equal bit for bit).  Planes of odd size and
smaller than one 16-byte piece, results that end inside a tile, every epilogue geometry, window instances, both types."""
import pytest
import torch

from heron_amd import backend as B
from heron_amd import hostops, instances
from heron_amd.ops.rocm import getOpFromName

pytestmark = pytest.mark.gpu

D, F16, U8, CONV = instances.D, instances.F16, instances.U8, instances.CONV
INSTANCES = {
    "f16-direct": D(F16, CONV, *instances.PARITY_SHAPES[2]),
    "f16-mfma16": D(F16, CONV, *instances.PARITY_SHAPES[5]),
    "f16-strips": D(F16, CONV, 128, 64, 64, 4, 1, 16, 3, 3, epi=1),
    "f16-window": D(F16, CONV, 64, 64, 64, 2, 2, 32, 2, 2, epi=1, win=1),
    "u8s8": instances.int8_conv_descs()[0],
    "u8s8-colsum": instances.int8_conv_descs()[6],
    "u8s8-window": instances.int8_conv_descs()[7],
    "u8s8-window-16-waves": instances.chw_room_descs()[0],      # strips of 64 pixels do not fit beside the stages
}
CASES = [
    ("c1d", [3, 33, 64, 24, 3, 1, 1, 1]), ("c1d", [2, 100, 24, 136, 1, 2, 0, 1]),
    ("c2d_nchw", [2, 9, 9, 64, 40, 3, 3, 1, 1, 1]), ("c2d_nchw", [5, 2, 1, 64, 8, 1, 1, 1, 0, 1]), ("c2d_nchw", [1, 16, 24, 20, 72, 3, 3, 2, 1, 1]),
    ("c3d", [2, 3, 7, 5, 16, 24, 3, 3, 3, 1, 1, 1]), ("c3d", [1, 4, 8, 8, 64, 64, 1, 1, 1, 2, 0, 1]),
    ("t2d", [2, 7, 5, 64, 24, 3, 3, 2, 1, 1, 0]), ("t2d", [1, 6, 6, 24, 40, 1, 1, 4, 0, 1, 0]), ("t2d", [2, 5, 5, 64, 16, 3, 3, 1, 1, 1, 0]),
    ("t2d", [2, 4, 6, 64, 16, 3, 3, 2, 0, 1, 1]),
]


class Ctx:
    def set_info(self, info):
        self.info = info

    def set_axis_map(self, m):
        pass


# input windows whose position is carried from load to load: images smaller than a load's step, pixels of 24 chunks (no power of
# two), one row or one column, a halo larger than the image, several images in a window
WINDOW_CASES = [
    ("t2d", [9, 2, 2, 64, 16, 1, 1, 2, 0, 1, 0]), ("t2d", [5, 1, 1, 64, 16, 3, 3, 2, 1, 1, 0]), ("t2d", [2, 9, 1, 192, 24, 3, 3, 4, 1, 1, 0]),
    ("t2d", [3, 3, 11, 192, 64, 3, 3, 2, 1, 1, 0]), ("t2d", [40, 1, 2, 64, 8, 1, 1, 1, 0, 1, 0]), ("t2d", [1, 17, 15, 128, 64, 3, 3, 2, 1, 1, 0]),
    ("c2d_nchw", [7, 3, 1, 192, 24, 3, 3, 1, 1, 1]), ("c2d_nchw", [2, 11, 13, 192, 64, 3, 3, 1, 1, 1]), ("c2d_nchw", [30, 1, 1, 64, 8, 5, 5, 1, 2, 1]),
]


@pytest.mark.parametrize("name,cases", [(n, CASES) for n in sorted(INSTANCES)] + [(n, WINDOW_CASES) for n in INSTANCES if "window" in n],
                         ids=sorted(INSTANCES) + [n + "-carry" for n in INSTANCES if "window" in n])
def test_equals_the_separate_passes(name, cases, hrn):
    f16 = name.startswith("f16")
    mod = B.Module(INSTANCES[name])
    ran = 0
    for op, args in cases:
        ctx = Ctx()
        getOpFromName(op)(ctx, *args, *(["float16"] * 2 if f16 else ["int8"] * 2))
        info, ref = ctx.info, ctx.info["reference_args"]
        c = info["conv"]
        if INSTANCES[name].conv_window and not (c["stride"] == c["stride_w"] == 1 and c["HO"] == c["H"] and c["WO"] == c["W"] and
                                                c["CI"] * (2 if f16 else 1) % INSTANCES[name].bkb == 0):
            continue
        gen = torch.Generator(device="cuda").manual_seed(len(op) + sum(args))
        if f16:
            X = torch.randn(ref["input"], device="cuda", generator=gen).half()
            F = torch.randn(ref["filter"], device="cuda", generator=gen).half()
        else:
            X = torch.randint(0, 256, ref["input"], device="cuda", generator=gen, dtype=torch.uint8)
            F = torch.randint(-128, 128, ref["filter"], device="cuda", generator=gen, dtype=torch.int8)
        print("channels first", name, op, args, flush=True)
        got = hostops.run_operator(mod, info, [X, F])
        act, const, fin = hostops.ADAPTERS[info["adapter"]]
        want = fin(info, hostops.conv2d_nhwc(mod, act(info, X, F), const(info, X, F), (c["stride"], c["stride_w"]), (c["pad"], c["pad_w"]),
                                             (c["dil"], c["dil_w"])))
        torch.cuda.synchronize()
        assert got.shape == want.shape and torch.equal(got, want), (name, op, args)
        ran += 1
    assert ran >= 2
    mod.close()


def test_bad_views_are_refused(hrn):
    mod = B.Module(INSTANCES["f16-direct"])
    x = torch.zeros((1, 4, 4, 64), device="cuda").half()
    w = torch.zeros((8, 1, 1, 64), device="cuda").half()
    out = torch.zeros((1, 8, 8, 8), device="cuda").half()
    p = B.conv2d_problem(1, 8, 8, 64, 8, 1, 1, 1, 0, 1)
    for view in (B.ConvView(0), B.ConvView(63), B.ConvView(64, 3, 2, 2, 0, 0), B.ConvView(64, 2, 5, 4, 0, 0), B.ConvView(64, 2, 4, 4, 2, 0),
                 B.ConvView(64, 2, 4, 4, -1, 0)):
        with pytest.raises(B.HeronRocmError):
            mod.launch_conv2d_chw(p, view, x.data_ptr(), w.data_ptr(), out.data_ptr(), 0)
    mod.close()
    split = B.Module(instances.splitk_descs()[4])
    with pytest.raises(B.HeronRocmError):
        split.launch_conv2d_chw(p, B.ConvView(64), x.data_ptr(), w.data_ptr(), out.data_ptr(), 0)
    split.close()
