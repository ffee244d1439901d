"""Split BF16 of small outputs (one launch, K shared out over the waves): the
sums of the hi parts and of the lo parts meet in one rounding."""
import pytest
import torch

from _helpers import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N,p", [(100, 2048, 70, 0.5), (64, 300, 64, 0.9), (500, 7000, 304, 0.2)])
def test_one_rounding(bws, dev, M, K, N, p):
    """b = i + j/256 with whole i in [129, 254] and |j| <= 127: RNE to BF16 gives
    hi = i (ulp 1) and lo = j/256, both exact.  Sums of up to 7000 i (21 bits) and
    of j/256 (20 bits) are exact in any order, their sum is not: it has to be the
    FP32 number nearest to the exact one."""
    A = bws.Bitmap(to_dev(bws.gen_bitmap_iid(M + K, M, K, p), dev), M, K)
    g = torch.Generator(device=dev).manual_seed(K)
    i = torch.randint(129, 255, (K, N), device=dev, generator=g)
    j = torch.randint(-127, 128, (K, N), device=dev, generator=g)
    B = i.double() + j.double() / 256
    assert torch.equal(B.float().bfloat16().double(), i.double())
    R = bws.unpack_bitmap(A).double() @ B
    assert torch.equal(bws.spmm(A, B.float(), "bf16x2"), R.float())
