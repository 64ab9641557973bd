"""Split-K launches give every XCD an eighth of the (tile, slice) pairs: each pair belongs to one workgroup, whatever the counts, and
results are right for counts that 8 does and does not divide."""
import pytest
import torch

from heron_amd import backend as B
from heron_amd import hostops, instances
from launch_args import library


@pytest.mark.parametrize("pairs", list(range(1, 40)) + [63, 64, 65, 252, 255, 256, 257, 1001])
def test_every_pair_once(pairs):
    pair_of = library().pair_of
    assert sorted(pair_of(b, pairs) for b in range(pairs)) == list(range(pairs))
    for xcd in range(min(8, pairs)):
        own = [pair_of(b, pairs) for b in range(xcd, pairs, 8)]
        assert own == list(range(own[0], own[0] + len(own)))


@pytest.mark.gpu
@pytest.mark.parametrize("which", [0, 1, 2, 3, 6])
@pytest.mark.parametrize("m,n", [(1, 64), (65, 68), (130, 200), (64, 512), (200, 452)])
def test_products(which, m, n, hrn):
    d = instances.splitk_descs()[which]
    f16 = d.dtype == instances.F16
    mod = B.Module(d)
    gen = torch.Generator(device="cuda").manual_seed(m * n)
    for split, k in ((1, 64), (2, 272), (3, 400), (7, 1040)):
        for batch in (1, 3):
            a, w = (batch, m, k), (batch, n, k)
            if f16:      # sums of k products of -1, 0, 1: exact in fp16
                A = torch.randint(-1, 2, a, device="cuda", generator=gen).half()
                W = torch.randint(-1, 2, w, device="cuda", generator=gen).half()
            else:
                A = torch.randint(0, 2, a, device="cuda", generator=gen).to(torch.uint8)
                W = torch.randint(-128, 128, w, device="cuda", generator=gen, dtype=torch.int8)
            print("split-K raster", d.as_tuple(), (batch, m, n, k), split, flush=True)
            C = hostops.gemm(mod, A, W, split_k=split)
            for b in range(batch):
                assert torch.equal(C[b].float(), A[b].float() @ W[b].float().t())
    mod.close()


@pytest.mark.gpu
@pytest.mark.parametrize("which", [4, 5])
@pytest.mark.parametrize("n,h,w,co", [(1, 5, 5, 64), (3, 6, 5, 192), (8, 8, 8, 64), (2, 9, 7, 128)])     # 1, 6, 8 and 4 tiles
def test_convs(which, n, h, w, co, hrn):
    d = instances.splitk_descs()[which]
    f16 = d.dtype == instances.F16
    mod = B.Module(d)
    gen = torch.Generator(device="cuda").manual_seed(n * h + co)
    X = torch.randint(-1 if f16 else 0, 2, (n, h, w, 80), device="cuda", generator=gen)
    W = torch.randint(-1, 2, (co, 3, 3, 80), device="cuda", generator=gen)
    want = torch.nn.functional.conv2d(X.cpu().float().permute(0, 3, 1, 2), W.cpu().float().permute(0, 3, 1, 2), padding=1).permute(0, 2, 3, 1)
    for split in (1, 2, 3, 5):      # sums of at most 720 products of -1, 0, 1: exact in fp16
        print("split-K raster", d.as_tuple(), (n, h, w, 80, co), split, flush=True)
        Y = hostops.conv2d_nhwc(mod, X.to(torch.float16 if f16 else torch.uint8), W.to(torch.float16 if f16 else torch.int8), 1, 1, 1, split_k=split)
        assert torch.equal(Y.cpu().float(), want), split
    mod.close()
