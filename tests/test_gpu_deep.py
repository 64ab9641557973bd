"""Launches small enough for a third stage (the deep kernels) against the same instance on a grid too large for it: same products
in the same order, equal bit for bit.  k-tiles at both sides of the rule, K that ends inside a k-tile, M and N that end
inside a tile, plain and staged epilogues, one, two and four k-steps per tile, split-K; the channels-first deep kernels
against the oracle.  Module.is_deep says which kernel a launch takes."""
import numpy as np
import pytest
import torch

import oracle
from heron_amd import backend as B
from heron_amd import hostops, instances
from heron_amd.ops.rocm import getOpFromName
from parity_checks import check_f16

pytestmark = pytest.mark.gpu

D, F16, U8, GEMM, CONV = instances.D, instances.F16, instances.U8, instances.GEMM, instances.CONV
INSTANCES = {
    "f16": D(F16, GEMM, 128, 128, 128, 2, 2, 32, 2, 1, nt=1),
    "u8s8": D(U8, GEMM, 128, 128, 128, 2, 2, 16, 2, 1, epi=1, colsum=1, nt=1),
    "u8s8-split": instances.splitk_descs()[3],
    "f16-one-step": instances.deep_descs()[0],
    "u8s8-one-step": instances.deep_descs()[1],
}


def _inputs(f16, b, m, n, k):
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    if f16:
        return (torch.randn((b, m, k), device="cuda", generator=gen).half(), torch.randn((b, n, k), device="cuda", generator=gen).half())
    return (torch.randint(0, 256, (b, m, k), device="cuda", generator=gen, dtype=torch.uint8),
            torch.randint(-128, 128, (b, n, k), device="cuda", generator=gen, dtype=torch.int8))


@pytest.mark.parametrize("name", sorted(INSTANCES))
@pytest.mark.parametrize("k_tiles", [5, 6, 7, 8, 33])
@pytest.mark.parametrize("rest", [0, 16, 112])
def test_equals_the_plain_kernel(name, k_tiles, rest, hrn):
    d = INSTANCES[name]
    mod, f16 = B.Module(d), d.dtype == F16
    m, n, slices = (1025, 1028, 3) if d.split_k else ((1700, 1732, 0) if d.bkb == 128 else (3100, 3300, 0))
    kb = (k_tiles * d.bkb - min(rest, d.bkb - 16)) * max(1, slices)
    assert (m + n) * kb >= 2 << 20 or k_tiles < 6
    batch = 4                                          # the tiles of 4 entries are too many for it, one entry's are not
    k = kb // (2 if f16 else 1)
    assert not mod.is_deep(B.gemm_problem(batch, m, n, k, split_k=slices))
    assert mod.is_deep(B.gemm_problem(1, m, n, k, split_k=slices)) == (k_tiles >= 6)
    A, W = _inputs(f16, batch, m, n, k)
    print("deep", name, k_tiles, rest, flush=True)
    plain = hostops.gemm(mod, A, W, split_k=slices)
    for i in (0, batch - 1):
        got = hostops.gemm(mod, A[i], W[i], split_k=slices)
        assert torch.equal(got, plain[i]), (name, k_tiles, rest, i)
    mod.close()


@pytest.mark.parametrize("dtype", ["f16", "u8s8"])
def test_conv_images_in_one_launch_and_apart(dtype, hrn):
    f16 = dtype == "f16"
    d = D(F16, CONV, 128, 64, 128, 2, 1, 32, 2, 1, epi=1) if f16 else instances.int8_conv_descs()[0]
    mod = B.Module(d)
    gen = torch.Generator(device="cuda").manual_seed(3)
    shape, filt = (16, 33, 31, 1024 if f16 else 2048), (72, 3, 3, 1024 if f16 else 2048)
    if f16:
        X, F = torch.randn(shape, device="cuda", generator=gen).half(), torch.randn(filt, device="cuda", generator=gen).half()
    else:
        X = torch.randint(0, 256, shape, device="cuda", generator=gen, dtype=torch.uint8)
        F = torch.randint(-128, 128, filt, device="cuda", generator=gen, dtype=torch.int8)
    print("deep conv", dtype, flush=True)
    for stride in (1, 2):
        one, many = (B.conv2d_problem(n, *shape[1:], *filt[:3], stride, 1, 1) for n in (1, 16 * shape[0]))
        assert mod.is_deep(one) and not mod.is_deep(many)
        apart = torch.cat([hostops.conv2d_nhwc(mod, X[i:i + 1], F, stride, 1, 1) for i in range(3)])
        assert torch.equal(apart, hostops.conv2d_nhwc(mod, torch.cat([X] * 16), F, stride, 1, 1)[:3])
    mod.close()


# two-stage im2col instances, and channels-first layers of at least 2 MB of operands on few tiles: k-tiles that end inside a
# tap, at a tap and inside the last one, planes of odd size, strides, depth, expansion with stride 1, 2 and 4
CHW_INSTANCES = {
    "f16": D(F16, CONV, *instances.PARITY_SHAPES[2]),
    "f16-one-step": instances.deep_descs()[2],
    "u8s8": instances.int8_conv_descs()[2],
}
CHW_CASES = [
    ("c1d", [8, 1001, 272, 72, 3, 1, 1, 1]), ("c2d_nchw", [16, 29, 27, 192, 64, 3, 3, 1, 1, 1]), ("c2d_nchw", [16, 33, 31, 144, 40, 3, 3, 2, 1, 1]),
    ("c3d", [8, 4, 9, 11, 256, 72, 3, 3, 3, 1, 1, 1]), ("t2d", [16, 14, 13, 192, 64, 3, 3, 2, 1, 1, 1]), ("t2d", [16, 8, 8, 144, 40, 3, 3, 4, 0, 1, 0]),
    ("t2d", [16, 29, 27, 192, 24, 3, 3, 1, 1, 1, 0]),
]


def _oracle(op, args, X, F):
    s, p, d = args[-4:-1] if op == "t2d" else args[-3:]
    if op == "c1d":
        return oracle.conv1d_ncw_ref(X, F, s, p, d)
    if op == "c2d_nchw":
        return oracle.conv2d_nchw_ref(X, F, s, p, d)
    return oracle.conv3d_ncdhw_ref(X, F, s, p, d) if op == "c3d" else oracle.conv2d_transposed_nchw_ref(X, F, s, p, d, args[-1])


@pytest.mark.parametrize("name", sorted(CHW_INSTANCES))
@pytest.mark.parametrize("op,args", CHW_CASES, ids=["%s-%d" % (o, i) for i, (o, _) in enumerate(CHW_CASES)])
def test_channels_first(name, op, args, hrn):
    mod, f16 = B.Module(CHW_INSTANCES[name]), name.startswith("f16")
    ctx = type("Ctx", (), dict(set_info=lambda self, i: setattr(self, "info", i), set_axis_map=lambda self, m: None))()
    getOpFromName(op)(ctx, *args, *(["float16"] * 2 if f16 else ["int8"] * 2))
    info, c = ctx.info, ctx.info["conv"]
    assert mod.has_chw and mod.is_deep(B.conv2d_problem(*(c[n] for n in ("N", "H", "W", "CI", "CO", "KH", "KW")), (c["stride"], c["stride_w"]),
                                                        (c["pad"], c["pad_w"]), (c["dil"], c["dil_w"])))
    rng = np.random.default_rng(sum(args))
    shapes = info["reference_args"]["input"], info["reference_args"]["filter"]
    if f16:
        X, F = (rng.normal(0, 1, s).astype(np.float16) for s in shapes)
    else:
        X, F = rng.integers(0, 256, shapes[0], dtype=np.uint8), rng.integers(-128, 128, shapes[1], dtype=np.int8)
    print("deep channels first", name, op, args, flush=True)
    got = hostops.run_operator(mod, info, [torch.from_numpy(X).cuda(), torch.from_numpy(F).cuda()]).cpu().numpy()
    want = _oracle(op, args, X, F)
    assert got.shape == want.shape
    if f16:
        check_f16(got, want)
    else:
        assert np.array_equal(got, want)
    mod.close()
