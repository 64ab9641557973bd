"""Instances with epilogue 0 take results of any alignment: rows that are no whole 16-byte pieces, results that start at any element,
M and N that end inside a tile and inside a piece, memory around the result untouched; equal bit for bit to the same
instance with epilogue 1 where that takes the problem."""
import numpy as np
import pytest
import torch

import oracle
from heron_amd import backend as B
from heron_amd import hostops, instances
from parity_checks import check_f16

pytestmark = pytest.mark.gpu

D, F16, U8, GEMM, CONV = instances.D, instances.F16, instances.U8, instances.GEMM, instances.CONV
PAIRS = [(F16, (128, 128, 128, 2, 2, 32, 2, 1)), (U8, (128, 128, 128, 2, 2, 32, 2, 1)), (U8, (64, 64, 64, 1, 2, 16, 2, 3)), (F16, (64, 64, 64, 1, 2, 16, 2, 3))]


@pytest.mark.parametrize("kind,shape", PAIRS)
@pytest.mark.parametrize("n", [4, 36, 100, 128, 132, 260])
def test_rows_and_starts(kind, shape, n, hrn):
    f16 = kind == F16
    mods = [B.Module(D(kind, GEMM, *shape, epi=e)) for e in (0, 1)]
    rng = np.random.default_rng(n)
    for m in (1, 127, 131):
        k = 160
        if f16:
            A, W = rng.normal(0, 1, (m, k)).astype(np.float16), rng.normal(0, 1, (n, k)).astype(np.float16)
        else:
            A, W = rng.integers(0, 256, (m, k), dtype=np.uint8), rng.integers(-128, 128, (n, k), dtype=np.int8)
        a, w = torch.from_numpy(A).cuda(), torch.from_numpy(W).cuda()
        for start in (0, 1, 2, 4):
            buf = torch.full((m * n + 64,), -3, dtype=torch.float16 if f16 else torch.int32, device="cuda")
            out = buf[16 + start:16 + start + m * n].view(m, n)
            print("direct epilogue", kind, shape, (m, n, k), start, flush=True)
            hostops.gemm(mods[0], a, w, out=out)
            assert (buf[:16 + start] == -3).all() and (buf[16 + start + m * n:] == -3).all()
            if f16:
                check_f16(out.cpu().numpy(), oracle.gemm_f32(A, W))
            else:
                assert np.array_equal(out.cpu().numpy(), oracle.gemm_int64_numpy(A, W).astype(np.int32))
            if n % 8 == 0 or not f16:
                assert torch.equal(out, hostops.gemm(mods[1], a, w))
    for mod in mods:
        mod.close()
