"""The one-launch FP32 product of a 0/1 mask (128 x 32 tiles, K shared out over
2, 4 or 8 waves, bitmap words through LDS 1024 per wave at a time): edges of
its tiles, its steps and its chunks of words, odd widths, unaligned words and
operands.  Bounds as in test_gpu_fp32_matrix."""
import pytest
import torch

from _helpers import to_dev
from test_gpu_fp32_matrix import _check, _mask

pytestmark = pytest.mark.gpu

# M and N at, below and past a tile; K at and past a step, a chunk of words (4096
# columns with four waves, 8192 with eight), a wave's share; every wave count
CASES = [(1, 128, 1, 1.0), (127, 129, 31, 0.3), (128, 160, 32, 0.5), (129, 255, 33, 0.2),
         (257, 8192, 2, 0.05), (130, 8193, 3, 0.05), (200, 8300, 1, 0.1), (70, 16500, 36, 0.02),
         (3300, 4097, 301, 0.05), (3201, 4128, 322, 0.03), (2048, 1024, 2048, 0.05),
         (2040, 1000, 1999, 0.3), (3100, 1027, 3103, 0.1)]


@pytest.mark.parametrize("M,K,N,p", CASES)
def test_edges(bws, dev, M, K, N, p):
    A, D = _mask(bws, dev, M, K, p, M + K + N)
    g = torch.Generator(device=dev).manual_seed(N)
    B = torch.randn((K, N), device=dev, generator=g)
    _check(bws.spmm(A, B), D, B, K)
    # integers that fit 24 bits: exact; rows off 16 bytes, alpha and beta
    Bi = torch.randint(-1000, 1001, (K, N + 3), device=dev, generator=g).float()[:, 1:N + 1]
    C0 = torch.randint(-9, 10, (M, N + 1), device=dev, generator=g).float()
    C = C0.clone()
    bws.spmm(A, Bi, alpha=-2.0, beta=3.0, out=C[:, :N])
    assert torch.equal(C[:, :N].double(), -2.0 * (D @ Bi.double()) + 3.0 * C0[:, :N].double())
    assert torch.equal(C[:, N], C0[:, N])


def test_words_off_16_bytes(bws, dev):
    """Rows of bitmap words that start off 16 bytes, with room past the last one."""
    M, K, N = 300, 1000, 200
    A, D = _mask(bws, dev, M, K, 0.2, 9)
    nw = A.words.shape[1]
    W = torch.full((1 + M * (nw + 5),), -1, dtype=torch.int32, device=dev)[1:].view(M, nw + 5)
    W[:, :nw] = A.words
    A2 = bws.Bitmap(W, M, K)
    B = torch.randint(-1000, 1001, (K, N), device=dev).float()
    assert torch.equal(bws.spmm(A2, B).double(), D @ B.double())


@pytest.mark.parametrize("M,K,N", [(300, 9000, 100), (3300, 4200, 301), (2048, 200, 1999)])
def test_special_values(bws, dev, M, K, N):
    """An infinity, a NaN and values below the parts' range reach the rows that
    select them and no other, with every wave count."""
    A, D = _mask(bws, dev, M, K, 0.01, 21)
    B = torch.randint(-1000, 1001, (K, N), device=dev).float()
    B[3, 1], B[K - 1, 2], B[:, 4] = float("inf"), float("nan"), 2.0 ** -130
    C = bws.spmm(A, B)
    hit1, hit2 = D[:, 3] != 0, D[:, K - 1] != 0
    assert torch.equal(torch.isinf(C[:, 1]), hit1) and torch.equal(torch.isnan(C[:, 2]), hit2)
    B[3, 1] = B[K - 1, 2] = 0.0
    R = D @ B.double()
    ok = torch.ones((M, N), dtype=torch.bool, device=dev)
    ok[:, 1], ok[:, 2] = ~hit1, ~hit2
    assert torch.equal(C.double()[ok], R[ok])
