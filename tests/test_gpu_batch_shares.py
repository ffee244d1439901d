"""Grouped launches share every problem's tiles over the XCDs: each tile is
computed once whatever its problem's tile count (below, at and past the eight
shares, several problems in rotation, K from one stage to many)."""
import pytest
import torch

from _helpers import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,N", [("bf16", 128), ("bf16", 264), ("fp32", 256), ("bf16x2", 130)])
def test_batch_shares(bws, dev, prec, N):
    g = torch.Generator(device=dev).manual_seed(N)
    dt = torch.bfloat16 if prec == "bf16" else torch.float32
    probs, want = [], []
    for i, (M, K) in enumerate([(1, 64), (100, 700), (128, 33), (500, 64), (1000, 300), (1100, 2000),
                                (1025, 1), (2050, 129), (64, 4096), (300, 64)]):
        A = bws.Bitmap(to_dev(bws.gen_bitmap_iid(i, M, K, 0.2), dev), M, K)
        # integers: every order of addition gives the same sum
        B = torch.randint(-8, 9, (K, N), device=dev, generator=g).to(dt)
        probs.append((A, B, torch.full((M, N), float("nan"), device=dev)))
        want.append(bws.unpack_bitmap(A).double() @ B.double())
    bws.spmm_batched(probs, prec)
    for (A, _, C), R in zip(probs, want):
        assert torch.equal(C.double(), R), (A.rows, A.cols)
