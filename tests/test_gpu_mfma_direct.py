"""16-bit products of small outputs with a long K (64 x 64 and 128 x 64 tiles, K
shared out over eight waves, bitmap words through LDS 16384 or 8192 columns at a
time): edges of tiles, steps and chunks, widths and rows of B at any alignment,
FP32 B rounded in registers.  Sums of K products in any order, each addition
rounded or truncated to 24 bits, are within K 2^-23 of sum |b|; sums of integers
that fit 24 bits are exact."""
import pytest
import torch

from _helpers import to_dev

pytestmark = pytest.mark.gpu

DT = {"bf16": torch.bfloat16, "fp16": torch.float16}
CASES = [(1, 1280, 1, 1.0), (63, 1300, 65, 0.3), (64, 16384, 64, 0.02), (65, 16390, 3, 0.1),
         (130, 16500, 2, 0.1), (1000, 1281, 1023, 0.05), (1100, 8192, 1090, 0.02),
         (1999, 8200, 1001, 0.1), (2047, 2049, 1022, 0.05), (129, 2100, 8000, 0.2)]


@pytest.mark.parametrize("M,K,N,p", CASES)
@pytest.mark.parametrize("prec", ["bf16", "fp16"])
def test_direct16(bws, dev, M, K, N, p, prec):
    A = bws.Bitmap(to_dev(bws.gen_bitmap_iid(M + N, M, K, p), dev), M, K)
    D = bws.unpack_bitmap(A).double()
    g = torch.Generator(device=dev).manual_seed(K)
    B = torch.randn((K, N), device=dev, generator=g)
    Bh = B.to(DT[prec])
    C = bws.spmm(A, Bh, prec)
    R, S = D @ Bh.double(), D @ Bh.double().abs()
    assert bool(((C - R).abs() <= (K + 4) * 2.0 ** -23 * S).all())
    assert torch.equal(C, bws.spmm(A, B, prec))  # FP32 B: rounded to the same values
    # integers: exact; rows of B and C off 16 bytes, alpha and beta
    Bi = torch.randint(-100, 101, (K, N + 3), device=dev, generator=g).to(DT[prec])[:, 1:N + 1]
    C0 = torch.randint(-9, 10, (M, N + 1), device=dev, generator=g).float()
    for b in (Bi, Bi.float()):
        C = C0.clone()
        bws.spmm(A, b, prec, alpha=-2.0, beta=3.0, out=C[:, :N])
        assert torch.equal(C[:, :N].double(), -2.0 * (D @ Bi.double()) + 3.0 * C0[:, :N].double())
        assert torch.equal(C[:, N], C0[:, N])


@pytest.mark.parametrize("M,K,N,p", [(1, 1, 1, 1.0), (63, 31, 65, 0.5), (65, 33, 3, 0.4),
                                     (130, 16500, 2, 0.1), (1000, 700, 1023, 0.1),
                                     (1100, 8200, 1090, 0.02), (2048, 100, 2047, 0.2)])
def test_direct_split(bws, dev, M, K, N, p):
    """BF16X2: both parts of an FP32 B, 16 bits of each value."""
    A = bws.Bitmap(to_dev(bws.gen_bitmap_iid(M + N, M, K, p), dev), M, K)
    D = bws.unpack_bitmap(A).double()
    g = torch.Generator(device=dev).manual_seed(K)
    B = torch.randn((K, N), device=dev, generator=g)
    R, S = D @ B.double(), D @ B.double().abs()
    C = bws.spmm(A, B, "bf16x2")
    assert bool(((C - R).abs() <= ((2 * K + 4) * 2.0 ** -23 + 2.0 ** -16) * S).all())
    # integers of 10 bits: exact; rows of B and C off 16 bytes, alpha and beta
    Bi = torch.randint(-1000, 1001, (K, N + 3), device=dev, generator=g).float()[:, 1:N + 1]
    C0 = torch.randint(-9, 10, (M, N + 1), device=dev, generator=g).float()
    C = C0.clone()
    bws.spmm(A, Bi, "bf16x2", alpha=-2.0, beta=3.0, out=C[:, :N])
    assert torch.equal(C[:, :N].double(), -2.0 * (D @ Bi.double()) + 3.0 * C0[:, :N].double())
    assert torch.equal(C[:, N], C0[:, N])
