"""hrn_pad_rows word by word: rows around multiples of 16 bytes, sources that start at any element and hold less than one
16-byte word, several words of padding, rows long enough for many blocks.  Copies: equal exactly."""
import pytest
import torch

from heron_amd import backend as B

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.uint8])
def test_words(dtype, hrn):
    es = dtype.itemsize
    v = 16 // es
    for c in (1, 2, v - 1, v, v + 1, 2 * v - 1, 3 * v, 129, 8191):
        for rows in (1, 2, 3, 300):
            for skip in (0, 1, 3):
                for extra in (0, 2 * v):
                    cp = -(-c // v) * v + extra
                    t = torch.randint(0, 200, (skip + rows * c,), device="cuda").to(dtype)[skip:]
                    out = torch.full((rows + 1, cp), 7, dtype=dtype, device="cuda")
                    B.pad_rows(t.data_ptr(), out.data_ptr(), rows, c, cp, es, torch.cuda.current_stream().cuda_stream)
                    assert torch.equal(out[:rows], torch.nn.functional.pad(t.view(rows, c), (0, cp - c))), (c, rows, skip, cp)
                    assert (out[rows] == 7).all()
