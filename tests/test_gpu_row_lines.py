"""Non-temporal instances store without the hint where rows of the result end inside memory lines: rows that end on lines, on half lines,
at 16 bytes and (epilogue 0) anywhere, results above and below 64 MiB, results that start inside a line, persistent launches."""
import pytest
import torch

from heron_amd import backend as B
from heron_amd import hostops, instances, tuned

pytestmark = pytest.mark.gpu

D, F16, U8, GEMM = instances.D, instances.F16, instances.U8, instances.GEMM
INSTANCES = {
    "f16-any": D(F16, GEMM, 128, 128, 128, 2, 2, 32, 2, 1, nt=1), "u8": D(U8, GEMM, 128, 128, 128, 2, 2, 16, 2, 1, epi=1, colsum=1, nt=1),
    "f16-halves": tuned.load("gemm_f16_8192").desc, "u8-halves": tuned.load("gemm_u8s8_8192").desc, "persistent": tuned.load("bmm_f16_qk").desc,
    "values": tuned.load("bmm_f16_pv").desc,
}


def _check(mod, b, m, n, k, start):
    f16 = mod.desc.dtype == F16
    gen = torch.Generator(device="cuda").manual_seed(n)
    if f16:      # sums of k products of small whole numbers: exact in fp16
        A = torch.randint(-3, 4, (b, m, k), device="cuda", generator=gen).half()
        W = torch.randint(-3, 4, (b, n, k), device="cuda", generator=gen).half()
    else:
        A = torch.randint(0, 256, (b, m, k), device="cuda", generator=gen, dtype=torch.uint8)
        W = torch.randint(-128, 128, (b, n, k), device="cuda", generator=gen, dtype=torch.int8)
    kind = torch.float16 if f16 else torch.int32
    buf = torch.full((b * m * n + 64 + start,), -7, dtype=kind, device="cuda")
    out = buf[32 + start:32 + start + b * m * n].view(b, m, n)
    print("row lines", mod.desc.as_tuple(), (b, m, n, k), start, flush=True)
    hostops.gemm(mod, A if b > 1 else A[0], W if b > 1 else W[0], out=out if b > 1 else out[0])
    for i in range(b):
        assert torch.equal(out[i].float(), A[i].float() @ W[i].float().t())      # (whole numbers below 2^24)
    assert (buf[:32 + start] == -7).all() and (buf[32 + start + b * m * n:] == -7).all()


@pytest.mark.parametrize("name", sorted(INSTANCES))
@pytest.mark.parametrize("n", [64, 96, 72, 128, 136, 16])
def test_rows(name, n, hrn):
    mod = B.Module(INSTANCES[name])
    e = 16 // (2 if mod.desc.dtype == F16 else 4)
    for b, m in ((1, 1), (1, 255), (3, 130)):
        for start in (0, e):
            _check(mod, b, m, n, 48, start)
    if mod.desc.epilogue == 0:
        _check(mod, 1, 129, n + 4, 48, 3)
    mod.close()


@pytest.mark.parametrize("name,m,n", [("u8", 4100, 4112), ("f16-halves", 8195, 4128), ("persistent", 8200, 4128)])
def test_half_lines_above_64_mib(name, m, n, hrn):
    mod = B.Module(INSTANCES[name])
    _check(mod, 1, m, n, 16, 0)
    mod.close()
