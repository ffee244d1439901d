"""The 16-bit tile chosen for an output: 64 x 128 while 512 of them run at once."""
import pytest
import torch

from _helpers import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,rows,cols", [(2048, 2048, 64, 128), (2048, 2056, 128, 128), (1280, 4096, 128, 128),
                                           (21824, 192, 128, 128), (1536, 2048, 64, 64), (1537, 2048, 64, 128),
                                           (256, 256, 32, 64)])
def test_tile(bws, dev, M, N, rows, cols):
    """As a grouped launch of one problem reports it; alone and grouped the sums are
    the same bits."""
    K = 300
    A = bws.Bitmap(to_dev(bws.gen_bitmap_iid(M, M, K, 0.2), dev), M, K)
    B = torch.randn((K, N), device=dev).bfloat16()
    C = torch.empty((M, N), device=dev)
    L = bws.spmm_batched([(A, B, C)], "bf16").launches[0]
    assert (L["rows"], L["cols"]) == (rows, cols)
    assert torch.equal(C, bws.spmm(A, B, "bf16"))
