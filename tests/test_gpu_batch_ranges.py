"""Grouped launches whose XCDs take ranges of the tiles (up to 256 tiles, or up to
eight a problem) and the ones beside them that take shares: every tile is
computed once, as the same problem alone has it."""
import pytest
import torch

from _helpers import to_dev

pytestmark = pytest.mark.gpu


def _offsets(bws, b, launch, count):
    """The launch's tile table in the workspace: (count + 1) offsets behind the
    problems (256-byte aligned)."""
    entry = 13 * 8
    start = (entry * count + 255) // 256 * 256
    return b.ws[start:start + 8 * (count + 1)].view(torch.int64).tolist()


@pytest.mark.parametrize("prec,dt,N", [("fp16", torch.float32, 100), ("bf16x2", torch.float32, 130),
                                       ("bf16", torch.bfloat16, 264), ("bf16", torch.bfloat16, 33),
                                       ("fp32", torch.float32, 256), ("vals", torch.float32, 256)])
@pytest.mark.parametrize("count,lo,hi", [(7, 1, 700), (40, 1, 900), (9, 3000, 4000), (66, 300, 400)])
def test_tiles_once(bws, dev, prec, dt, N, count, lo, hi):
    g = torch.Generator(device=dev).manual_seed(N)
    probs, want = [], []
    for i in range(count):
        M, K = lo + (i * 397) % (hi - lo), 1 + (i * 211) % 400
        A = bws.Bitmap(to_dev(bws.gen_bitmap_iid(i, M, K, 0.2), dev), M, K)
        D = bws.unpack_bitmap(A).double()
        if prec == "vals":
            rp = bws.row_ptr(A)
            v = torch.randint(1, 9, (max(int(rp[-1]), 1),), device=dev, generator=g).float()
            A = A.with_values(v, rp)
            D[D != 0] = v[:int(rp[-1])].double()
        # integers: every order of addition gives the same sum
        B = torch.randint(-8, 9, (K, N), device=dev, generator=g).to(dt)
        probs.append((A, B, torch.full((M, N), float("nan"), device=dev)))
        want.append(D @ B.double())
    b = bws.spmm_batched(probs, "fp32" if prec == "vals" else prec)
    for (A, _, C), R in zip(probs, want):
        assert torch.equal(C.double(), R), (A.rows, A.cols)
    if len(b.launches) == 1 and b.launches[0]["kind"] != 3:
        L = b.launches[0]
        off = _offsets(bws, b, L, count)
        ranges = L["tiles"] <= max(256, 8 * count)
        assert (off[-1] == L["tiles"]) == ranges and off == sorted(off)
