"""The 16-bit tile chosen without a plan: 64 x 128 for one output while 512 of them
run at once, for a grouped launch up to 1280 tiles of 64 x 64."""
import pytest
import torch

from _helpers import to_dev

pytestmark = pytest.mark.gpu


def _problem(bws, dev, M, K, N):
    A = bws.Bitmap(to_dev(bws.gen_bitmap_iid(M, M, K, 0.2), dev), M, K)
    return A, torch.randn((K, N), device=dev).bfloat16(), torch.empty((M, N), device=dev)


@pytest.mark.parametrize("M,N,rows,cols", [(2048, 2048, 64, 128), (1280, 4096, 64, 128), (1281, 4096, 128, 128),
                                           (21824, 192, 64, 128), (1536, 2048, 64, 64), (1537, 2048, 64, 128),
                                           (256, 256, 32, 64)])
def test_grouped(bws, dev, M, N, rows, cols):
    """As the launch reports it; alone and grouped the sums are the same bits."""
    A, B, C = _problem(bws, dev, M, 300, N)
    L = bws.spmm_batched([(A, B, C)], "bf16").launches[0]
    assert (L["rows"], L["cols"]) == (rows, cols)
    assert torch.equal(C, bws.spmm(A, B, "bf16"))


def _us(f):
    best = 1e9
    for _ in range(7):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(12):
            f()
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b))
    return best


@pytest.mark.parametrize("M,N", [(2048, 2112), (4096, 1280)])
def test_alone(bws, dev, M, N):
    """More than 512 tiles of 64 x 128: within 6% of the 128 x 128 tiles that a plan
    selects (64 x 128, in two rounds, took 10 to 13% more)."""
    A, B, C = _problem(bws, dev, M, 2048, N)
    plan = bws.make_plan(2, rows_per_wg=128, cols_per_wg=128)
    assert _us(lambda: bws.spmm(A, B, "bf16", out=C)) <= \
        1.06 * _us(lambda: bws.spmm(A, B, "bf16", out=C, plan=plan))
