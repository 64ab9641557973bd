"""Edges of the register-block transpose (hrn_transpose_pad): widths and heights around one 16-byte piece and around the
64- and 128-element tiles, every remainder of a piece, padded and ragged result rows, in the three element sizes."""
import pytest
import torch

from heron_amd import backend as B

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.uint8, torch.float16, torch.int32])
def test_edges(dtype, hrn):
    st = torch.cuda.current_stream().cuda_stream
    v = 16 // torch.empty(0, dtype=dtype).element_size()
    shapes = [(1, r, c, r) for r in (1, v - 1, v, v + 1, 8 * v + 1) for c in (1, v - 1, v, v + 1, 8 * v - 1, 8 * v + 3)]
    shapes += [(3, 2 * v + e, 4 * v + e, 3 * v + 1) for e in range(v)]
    shapes += [(2, 5, 3 * v + 2, 2 * v), (5, 8 * v, 16 * v, 9 * v)]
    for b, r, c, rp in shapes:
        x = torch.randint(0, 120, (b, r, c), device="cuda").to(dtype)
        out = torch.full((b, c, rp), 9, dtype=dtype, device="cuda")
        print("transpose", dtype, b, r, c, rp, flush=True)
        B.transpose_pad(x.data_ptr(), out.data_ptr(), b, r, c, rp, x.element_size(), st)
        torch.cuda.synchronize()
        assert torch.equal(out, torch.nn.functional.pad(x.permute(0, 2, 1), (0, rp - r))), (dtype, b, r, c, rp)


@pytest.mark.parametrize("dtype", [torch.uint8, torch.float16, torch.int32])
def test_more_rows_than_one_grid_dimension_of_tiles(dtype, hrn):
    rows, cols = 65535 * 64 + 9, 3
    x = torch.randint(0, 120, (rows, cols), device="cuda").to(dtype)
    for rp in (rows, rows + 7):
        out = torch.full((cols, rp), 9, dtype=dtype, device="cuda")
        print("transpose", dtype, rows, cols, rp, flush=True)
        B.transpose_pad(x.data_ptr(), out.data_ptr(), 1, rows, cols, rp, x.element_size(), torch.cuda.current_stream().cuda_stream)
        assert torch.equal(out, torch.nn.functional.pad(x.t(), (0, rp - rows)))
