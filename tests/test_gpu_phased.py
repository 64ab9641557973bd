"""The phased schedule of the 256x256 tiles: K from one chunk over one, two and three k-tiles to a ragged last one, M and N
around the tile edge, both wave grids and both MFMA shapes in either element type, against the host references (uint8
bit-exact)."""
import numpy as np
import pytest
import torch

import oracle
from heron_amd import backend as B
from heron_amd import hostops, instances, tuned, workloads
from parity_checks import check_f16

pytestmark = pytest.mark.gpu

D, F16, U8, GEMM = instances.D, instances.F16, instances.U8, instances.GEMM
INSTANCES = {
    "f16-4x2": D(F16, GEMM, 256, 256, 128, 4, 2, 16, 2, 1, epi=2, sched=2),
    "f16-2x4": D(F16, GEMM, 256, 256, 128, 2, 4, 16, 2, 2),
    "u8s8-2x4": D(U8, GEMM, 256, 256, 128, 2, 4, 16, 2, 1, colsum=1),
    "u8s8-4x2": instances.phased_descs()[0],
    "u8s8-4x2-32x32": instances.phased_descs()[1],
    "u8s8-2x4-32x32": instances.phased_descs()[2],
    "f16-2x4-32x32": instances.phased_descs()[3],
    "f16-4x2-32x32": instances.phased_descs()[4],
    "u8s8-tuned": tuned.load("gemm_u8s8_8192").desc,
    "f16-tuned": tuned.load("gemm_f16_8192").desc,
}


@pytest.mark.parametrize("name", sorted(INSTANCES))
@pytest.mark.parametrize("kb", [16, 128, 144, 256, 272, 384, 400, 1024, 1040])
def test_k_tiles(name, kb, hrn):
    f16 = name.startswith("f16")
    mod = B.Module(INSTANCES[name])
    K = kb // 2 if f16 else kb
    for M, N in [(256, 256), (257, 264), (13, 520), (700, 248)]:
        A, Bm = (workloads.gemm_f16_inputs if f16 else workloads.gemm_u8s8_inputs)(M, K, N, seed=kb + M)
        print("phased", name, M, K, N, flush=True)
        C = hostops.gemm(mod, torch.from_numpy(A).cuda(), torch.from_numpy(Bm).cuda()).cpu().numpy()
        if f16:
            check_f16(C, oracle.gemm_f32(A, Bm))
        else:
            assert np.array_equal(C, oracle.gemm_int64_numpy(A, Bm).astype(np.int32))
    mod.close()
