"""Split-K launches that add their slices up themselves against the ones that leave it to a second launch: the same bits, whatever
the workspace held before, over edges of tiles, one slice to more than chains, few and many 16-byte pieces per tile."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from heron_amd import backend as B
from heron_amd import hostops, instances, workloads
from parity_checks import check_f16

pytestmark = pytest.mark.gpu

GEMMS = [d for d in instances.splitk_descs() if d.op == instances.GEMM]


def _problem(desc, b, M, N, K, split, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if desc.dtype == instances.F16:
        A, W = (torch.randn(b, r, K, device="cuda", generator=gen).half() * 0.1 for r in (M, N))
    else:
        A = torch.randint(0, 256, (b, M, K), dtype=torch.uint8, device="cuda", generator=gen)
        W = torch.randint(-128, 128, (b, N, K), dtype=torch.int8, device="cuda", generator=gen)
    p = B.gemm_problem(b, M, N, K, 8, split_k=split)
    bsum = hostops.column_sums(W) if desc.colsum else None
    if bsum is not None:
        p.bsum = bsum.data_ptr()
    return A, W, p, bsum


def _launch(mod, p, A, W, ws, size, fill):
    out = torch.full((A.shape[0], A.shape[1], W.shape[1]), -7, device="cuda", dtype=torch.float16 if A.dtype == torch.float16 else torch.int32)
    ws.fill_(fill)
    p.workspace, p.workspace_bytes = ws.data_ptr(), size
    f = B.lib().hrn_launch_bmm_f16 if A.dtype == torch.float16 else B.lib().hrn_launch_bmm_u8s8
    assert f(mod._h, ctypes.byref(p), A.data_ptr(), W.data_ptr(), out.data_ptr(), torch.cuda.current_stream().cuda_stream) == B.HRN_OK
    return out


# (batch, M, N, K, slices): whole tiles, remainders, one column piece, one row, more slices than the 8 chains, one slice
SHAPES = [(1, 128, 128, 1024, 4), (1, 65, 68, 2064, 7), (2, 1, 4, 4096, 16), (1, 3, 60, 1040, 2), (1, 33, 32, 8192, 61),
          (1, 64, 12, 8192, 64), (3, 130, 36, 512, 1), (1, 200, 200, 2048, 9)]


@pytest.mark.parametrize("desc", GEMMS, ids=lambda d: str(d.as_tuple()))
def test_same_bits_as_a_second_launch(desc, hrn):
    mod = B.Module(desc)
    for i, (b, M, N, K, split) in enumerate(SHAPES):
        print("split-K fold", desc.as_tuple(), (b, M, N, K, split), flush=True)
        A, W, p, bsum = _problem(desc, b, M, N, K, split, 40 + i)
        plain, fast = B.splitk_workspace_bytes(desc, p), B.splitk_workspace_bytes(desc, p, fast=True)
        tiles = -(-M // desc.bm) * -(-N // desc.bn) * b
        assert fast == plain + 8 * tiles
        ws = torch.empty(fast, dtype=torch.uint8, device="cuda")
        want = _launch(mod, p, A, W, ws, plain, 0)
        for fill in (0, 255, 1):                       # (and the words of the launch before lie where this one's are)
            assert torch.equal(_launch(mod, p, A, W, ws, fast, fill), want)
        got = hostops.gemm(mod, A, W, split_k=split, bsum=bsum)
        assert torch.equal(got, want)
        for e in range(b):
            if desc.dtype == instances.F16:
                check_f16(got[e].cpu().numpy(), oracle.gemm_f32(A[e].cpu().numpy(), W[e].cpu().numpy()))
            else:
                assert np.array_equal(got[e].cpu().numpy(), oracle.gemm_int64_numpy(A[e].cpu().numpy(), W[e].cpu().numpy()).astype(np.int32))
    mod.close()


def test_replays_of_a_graph(hrn):
    """A captured launch counts its arrivals anew in every replay, also with another launch in its workspace's words between."""
    desc = GEMMS[0]
    mod = B.Module(desc)
    A, W, p, _ = _problem(desc, 1, 96, 160, 2048, 5, 7)
    fast = B.splitk_workspace_bytes(desc, p, fast=True)
    ws = torch.zeros(fast, dtype=torch.uint8, device="cuda")
    want = _launch(mod, p, A, W, ws, fast, 0)
    out = torch.empty_like(want)
    f = B.lib().hrn_launch_bmm_f16
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        for _ in range(2):
            assert f(mod._h, ctypes.byref(p), A.data_ptr(), W.data_ptr(), out.data_ptr(), torch.cuda.current_stream().cuda_stream) == B.HRN_OK
    for step in range(4):
        A.mul_(-0.5)
        out.fill_(3)
        graph.replay()
        torch.cuda.synchronize()
        got = out.clone()
        assert torch.equal(got, _launch(mod, p, A, W, ws, fast, 255 if step % 2 else 0))
    mod.close()


def test_streams_and_problems_side_by_side(hrn):
    """Launches on two streams, each with a workspace of its own, and problems of other sizes through one workspace."""
    desc = GEMMS[0]
    mod = B.Module(desc)
    probs = [_problem(desc, 1, M, N, K, s, 60 + s) for M, N, K, s in [(64, 512, 4096, 6), (200, 128, 2048, 3), (16, 1024, 4096, 9)]]
    want = [hostops.gemm(mod, A, W, split_k=p.split_k).clone() for A, W, p, _ in probs]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    got = []
    for r in range(20):
        for st in streams:
            with torch.cuda.stream(st):
                got.append([hostops.gemm(mod, A, W, split_k=p.split_k) for A, W, p, _ in probs])
    torch.cuda.synchronize()
    for g in got:
        for a, b in zip(g, want):
            assert torch.equal(a, b)
    mod.close()
