"""hrn_gather_nd's index arithmetic: extents and divisors around powers of two and the remainders of both, up to all six
dimensions, 16-byte pieces and single elements.  Copies: equal exactly."""
import pytest
import torch

from heron_amd import backend as B

pytestmark = pytest.mark.gpu


def _run(src, dst_dim, coords):
    out = torch.full(dst_dim, 7, dtype=src.dtype, device="cuda")
    B.gather_nd(B.make_gather(src.element_size(), dst_dim, coords), src.data_ptr(), out.data_ptr(),
                stream=torch.cuda.current_stream().cuda_stream)
    return out


@pytest.mark.parametrize("dtype", [torch.uint8, torch.float16, torch.int32])
@pytest.mark.parametrize("inner", [1, 3, 16, 48])
@pytest.mark.parametrize("step", [1, 2, 3, 4, 7, 127, 128, 129])
def test_expansion(dtype, inner, step, hrn):
    """row y of the result is row (y - 2) / step of the source where that divides, else zero"""
    for rows in (1, 2, 31, 65):
        src = torch.randint(0, 100, (rows, inner), device="cuda").to(dtype)
        n = (rows - 1) * step + 5
        want = torch.zeros((n, inner), dtype=dtype, device="cuda")
        want[2:2 + (rows - 1) * step + 1:step] = src
        assert torch.equal(_run(src, (n, inner), [(rows, inner, {0: 1}, -2, step), (inner, 1, {1: 1})]), want), rows


@pytest.mark.parametrize("dims", [(2, 3, 5, 7, 9, 16), (1, 1, 257, 1, 3, 8), (255, 1, 17, 2, 1, 24), (3, 1, 1, 65537, 1, 1), (1, 1, 1, 1, 1, 1)])
def test_six_dimensions(dims, hrn):
    """a permutation of five dimensions with the innermost kept"""
    order = (3, 1, 4, 0, 2, 5)
    src = torch.randint(0, 30000, [dims[o] for o in order], device="cuda").half()
    coords = [(dims[o], src.stride(i), {o: 1}) for i, o in enumerate(order)]
    inverse = [order.index(d) for d in range(6)]
    assert torch.equal(_run(src, dims, coords), src.permute(*inverse).contiguous())
