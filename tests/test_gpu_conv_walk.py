"""im2col kernels against the definition where the offsets they carry along K and from row to row are hardest: channels at, above and no
multiple of a k-tile, unequal strides and dilations, filters of one and several columns, K slices that begin inside a filter row,
channels-first results and zero-expanded inputs; and strides, pads and dilations far larger than the image."""
import pytest
import torch

from heron_amd import backend as B
from heron_amd import hostops, instances

pytestmark = pytest.mark.gpu

D, F16, U8, CONV = instances.D, instances.F16, instances.U8, instances.CONV
INSTANCES = {
    "f16": D(F16, CONV, 128, 64, 128, 2, 1, 32, 2, 1, epi=1), "f16-64": D(F16, CONV, 128, 64, 64, 4, 1, 16, 3, 3, epi=1),
    "u8": D(U8, CONV, 128, 64, 128, 2, 2, 16, 3, 1, epi=1), "u8-64": instances.int8_conv_descs()[0],
}
SPLIT = {"f16": instances.splitk_descs()[4], "u8": instances.splitk_descs()[5]}
# n, h, w, kh, kw, co, (height, width) pairs of stride, pad and dilation
CONVS = [
    (2, 13, 17, 3, 3, 64, (1, 1), (2, 1), (2, 1)), (2, 13, 17, 3, 3, 64, (2, 1), (1, 3), (1, 3)), (3, 9, 11, 3, 1, 40, (1, 2), (3, 0), (3, 1)),
    (1, 19, 8, 2, 5, 64, (3, 1), (0, 4), (4, 2)), (5, 3, 2, 1, 3, 64, (1, 1), (0, 2), (1, 2)), (9, 2, 3, 1, 1, 16, (2, 2), (0, 0), (1, 1)),
]
CHANNELS = {"f16": [64, 72, 112, 200], "f16-64": [32, 40, 72, 104], "u8": [128, 144, 176, 272], "u8-64": [64, 80, 144, 176]}


def _operands(f16, n, h, w, ci, kh, kw, co):
    """Whole numbers whose sums are exact in every type of the way."""
    gen = torch.Generator().manual_seed(n * h + w * ci + kh * kw + co)
    x = torch.randint(-1 if f16 else 0, 2 if f16 else 4, (n, h, w, ci), generator=gen)
    f = torch.randint(-1, 2, (co, kh, kw, ci), generator=gen) * (torch.rand((co, kh, kw, ci), generator=gen) < 0.2)
    return x, f


def _reference(x, f, s, p, d):
    n, h, w, ci = x.shape
    co, kh, kw, _ = f.shape
    ho, wo = (h + 2 * p[0] - (kh - 1) * d[0] - 1) // s[0] + 1, (w + 2 * p[1] - (kw - 1) * d[1] - 1) // s[1] + 1
    out = torch.zeros((n, ho, wo, co))
    for r in range(kh):
        for c in range(kw):
            for oy in range(ho):
                iy = oy * s[0] - p[0] + r * d[0]
                cols = [(ox, ox * s[1] - p[1] + c * d[1]) for ox in range(wo)]
                cols = [(ox, ix) for ox, ix in cols if 0 <= ix < w]
                if 0 <= iy < h and cols:
                    out[:, oy, [ox for ox, _ in cols]] += x[:, iy, [ix for _, ix in cols]].float() @ f[:, r, c].float().t()
    return out


def _run(desc, x, f, s, p, d, split=0):
    mod = B.Module(desc)
    kinds = (torch.float16, torch.float16) if desc.dtype == F16 else (torch.uint8, torch.int8)
    print("conv walk", desc.as_tuple(), tuple(x.shape), tuple(f.shape), s, p, d, split, flush=True)
    y = hostops.conv2d_nhwc(mod, x.to(kinds[0]).cuda(), f.to(kinds[1]).cuda(), s, p, d, split_k=split).cpu()
    mod.close()
    return y.float()


@pytest.mark.parametrize("name", sorted(INSTANCES))
@pytest.mark.parametrize("conv", CONVS)
def test_channels_and_dilations(name, conv, hrn):
    n, h, w, kh, kw, co, s, p, d = conv
    for ci in CHANNELS[name]:
        x, f = _operands(name.startswith("f16"), n, h, w, ci, kh, kw, co)
        assert torch.equal(_run(INSTANCES[name], x, f, s, p, d), _reference(x, f, s, p, d)), ci


@pytest.mark.parametrize("name", sorted(SPLIT))
@pytest.mark.parametrize("conv", CONVS)
def test_slices_inside_a_filter_row(name, conv, hrn):
    n, h, w, kh, kw, co, s, p, d = conv
    for ci in (24, 72, 200) if name == "f16" else (48, 80, 176):
        x, f = _operands(name == "f16", n, h, w, ci, kh, kw, co)
        want = _reference(x, f, s, p, d)
        for split in (2, 3, 7):
            assert torch.equal(_run(SPLIT[name], x, f, s, p, d, split), want), (ci, split)


@pytest.mark.parametrize("name", sorted(INSTANCES))
@pytest.mark.parametrize("conv", [c for c in CONVS if c[6] == (1, 1)])
@pytest.mark.parametrize("expand", [0, 2, 4])
def test_channels_first(name, conv, expand, hrn):
    n, h, w, kh, kw, co, s, p, d = conv
    desc = INSTANCES[name]
    f16 = desc.dtype == F16
    mod = B.Module(desc)
    for ci in CHANNELS[name]:
        x, f = _operands(f16, n, h, w, ci, kh, kw, co)
        small = x
        if expand:
            top, left = min(1, h - 1), 0
            small = x[:, :(h - top - 1) // expand + 1, :(w - left - 1) // expand + 1].contiguous()
            x = torch.zeros_like(x)
            x[:, top::expand, left::expand] = small
        want = _reference(x, f, s, p, d)
        plane = want.shape[1] * want.shape[2]
        prob = B.conv2d_problem(n, h, w, ci, co, kh, kw, s, p, d)
        view = B.ConvView(plane, expand, small.shape[1], small.shape[2], top, left) if expand else B.ConvView(plane)
        X = small.to(torch.float16 if f16 else torch.uint8).cuda()
        F = f.to(torch.float16 if f16 else torch.int8).cuda()
        out = torch.full((n, co, plane), -7, dtype=torch.float16 if f16 else torch.int32, device="cuda")
        print("conv walk, channels first", desc.as_tuple(), tuple(x.shape), tuple(f.shape), s, p, d, expand, flush=True)
        mod.launch_conv2d_chw(prob, view, X.data_ptr(), F.data_ptr(), out.data_ptr(), 0)
        torch.cuda.synchronize()
        assert torch.equal(out.cpu().float(), want.reshape(n, plane, co).transpose(1, 2)), ci
    mod.close()


G = 1 << 30


@pytest.mark.parametrize("conv", [
    (2, 9, 9, 1, 1, 16, (1 << 26, 1 << 26), (0, 0), (1, 1)), (3, 5, 7, 3, 3, 16, (G, 2 * G - 1), (1, 1), (1, 1)),
    (2, 1, 1, 1, 1, 16, (G, G), (G, G), (1, 1)),                                # three rows of three, the image in the middle
    (2, 3, 3, 2, 2, 16, (G // 2, G // 2), (G // 2, G // 2), (G, G)), (1, 4, 4, 3, 3, 16, (G // 2, G // 2), (G // 2, G // 2), (G // 2, G // 2)),
    (4, 6, 6, 1, 1, 16, (2, 2), (0, 0), (G, 2 * G - 1)),
])
def test_far_strides_pads_and_dilations(conv, hrn):
    n, h, w, kh, kw, co, s, p, d = conv
    for name, ci in (("f16", 64), ("f16", 72), ("u8", 48)):
        x, f = _operands(name == "f16", n, h, w, ci, kh, kw, co)
        want = _reference(x, f, s, p, d)
        assert torch.equal(_run(INSTANCES[name], x, f, s, p, d), want)
        assert torch.equal(_run(SPLIT[name], x, f, s, p, d, 2), want)
