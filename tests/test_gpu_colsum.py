"""hrn_colsum_s8 at the row lengths where the lanes per row change, with the row counts of partly filled blocks, one matrix and
batches that do or do not follow one another, padded rows.  Whole numbers: equal exactly, nothing written past the sums."""
import pytest
import torch

from heron_amd import backend as B

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [16, 48, 64, 80, 128, 144, 256, 272, 512, 528, 1024, 1040, 2064])
def test_lanes_per_row(k, hrn):
    for batch, n in ((1, 1), (1, 65), (1, 257), (3, 7), (5, 64), (2, 1031)):
        for ldb in (k, k + 32):
            for gap in (0, 48):
                stride = n * ldb + gap
                t = torch.randint(-128, 128, (batch * stride,), dtype=torch.int8, device="cuda")
                out = torch.full((batch * n + 8,), 7, dtype=torch.int32, device="cuda")
                B.colsum_s8(t.data_ptr(), out.data_ptr(), batch, n, k, ldb, stride, torch.cuda.current_stream().cuda_stream)
                rows = t.view(batch, stride)[:, :n * ldb].reshape(batch, n, ldb)[:, :, :k]
                assert torch.equal(out[:batch * n], rows.sum(-1, dtype=torch.int32).flatten()), (batch, n, ldb, gap)
                assert (out[batch * n:] == 7).all()
