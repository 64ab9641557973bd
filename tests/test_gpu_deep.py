"""Launches small enough for a third stage (the deep kernels) against the same instance on a grid too large for it: same products
in the same order, equal bit for bit.  k-tiles at both sides of the rule, K that ends inside a k-tile, M and N that end
inside a tile, plain and staged epilogues, one and two k-steps per tile, split-K."""
import pytest
import torch

from heron_amd import backend as B
from heron_amd import hostops, instances

pytestmark = pytest.mark.gpu

D, F16, U8, GEMM, CONV = instances.D, instances.F16, instances.U8, instances.GEMM, instances.CONV
INSTANCES = {
    "f16": D(F16, GEMM, 128, 128, 128, 2, 2, 32, 2, 1, nt=1),
    "u8s8": D(U8, GEMM, 128, 128, 128, 2, 2, 16, 2, 1, epi=1, colsum=1, nt=1),
    "u8s8-split": instances.splitk_descs()[3],
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
    m, n, slices = (1025, 1028, 3) if d.split_k else (1700, 1732, 0)
    kb = (k_tiles * 128 - rest) * max(1, slices)
    assert (m + n) * kb >= 2 << 20 or k_tiles < 6
    batch = 4                                          # 4 x 196 (split: 4 x 459) tiles are too many, one entry's are not
    A, W = _inputs(f16, batch, m, n, kb // (2 if f16 else 1))
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
        apart = torch.cat([hostops.conv2d_nhwc(mod, X[i:i + 1], F, stride, 1, 1) for i in range(3)])
        assert torch.equal(apart, hostops.conv2d_nhwc(mod, torch.cat([X] * 16), F, stride, 1, 1)[:3])
    mod.close()
