"""16-bit products of small outputs (32 x 64, 64 x 64 and 64 x 128 tiles, 128-row
K stages) and of a B whose rows the direct copies cannot take (padded in the
workspace): the same bits as the 128 x 128 tile with registers between, which
walks K in the same order; grouped launches with the same tiles."""
import pytest
import torch

from _helpers import to_dev

pytestmark = pytest.mark.gpu

DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "bf16x2": torch.float32}


def _mask(bws, dev, M, K, p, seed):
    return bws.Bitmap(to_dev(bws.gen_bitmap_iid(seed, M, K, p), dev), M, K)


# every tile's range of outputs (up to 256, 768 and 1280 tiles of 64 x 64), edges
# of rows, columns and K stages
SHAPES = [(1, 1, 8, 1.0), (33, 127, 64, 0.5), (31, 129, 72, 0.3), (1000, 128, 1000, 0.1),
          (2049, 257, 520, 0.1), (130, 1000, 8200, 0.05), (4100, 300, 1032, 0.02)]


@pytest.mark.parametrize("M,K,N,p", SHAPES)
@pytest.mark.parametrize("prec", ["bf16", "fp16"])
def test_small_tiles(bws, dev, M, K, N, p, prec):
    A = _mask(bws, dev, M, K, p, M + N)
    g = torch.Generator(device=dev).manual_seed(K)
    B = torch.randn((K, N + 8), device=dev, generator=g).to(DT[prec])[:, 8:]
    plan = bws.make_plan(kernel=2, rows_per_wg=128, cols_per_wg=128, mfma_staging="regs")
    assert torch.equal(bws.spmm(A, B, prec), bws.spmm(A, B, prec, plan=plan))
    C0 = torch.randn((M, N + 4), device=dev, generator=g)
    C1, C2 = C0.clone(), C0.clone()
    bws.spmm(A, B, prec, alpha=0.5, beta=-2.0, out=C1[:, 2:N + 2])
    bws.spmm(A, B, prec, alpha=0.5, beta=-2.0, out=C2[:, 2:N + 2], plan=plan)
    assert torch.equal(C1, C2)


@pytest.mark.parametrize("M,K,N,p", [(5, 3, 2, 0.9), (100, 70, 1, 0.5), (257, 97, 130, 0.3),
                                     (1000, 500, 303, 0.05), (300, 129, 7, 0.2)])
@pytest.mark.parametrize("prec", ["bf16", "fp16", "bf16x2"])
@pytest.mark.parametrize("f32", [False, True])
def test_padded_rows(bws, dev, M, K, N, p, prec, f32):
    A = _mask(bws, dev, M, K, p, M + N)
    g = torch.Generator(device=dev).manual_seed(K)
    B = torch.randn((K, N + 3), device=dev, generator=g)
    B = (B if f32 or prec == "bf16x2" else B.to(DT[prec]))[:, 1:N + 1]
    plan = bws.make_plan(kernel=2, rows_per_wg=128, cols_per_wg=128, mfma_staging="regs")
    C, R = bws.spmm(A, B, prec), bws.spmm(A, B, prec, plan=plan)
    if prec == "bf16x2":  # two passes: one more rounding of the partial sum
        S = bws.unpack_bitmap(A).double() @ B.double().abs()
        assert bool(((C - R).double().abs() <= 2e-6 * S).all())
    else:
        assert torch.equal(C, R)


def test_misaligned_16bit_rows(bws, dev):
    """N a multiple of 8 but rows off 16 bytes."""
    A = _mask(bws, dev, 300, 200, 0.2, 1)
    big = torch.randn((200, 140), device=dev).to(torch.bfloat16)
    for B in (big[:, 1:129], big[:, :136]):
        assert torch.equal(bws.spmm(A, B, "bf16"), bws.spmm(A, B.contiguous(), "bf16"))


@pytest.mark.parametrize("sizes,N", [([(64, 64), (100, 300), (1, 5)], 64),         # 32 x 64
                                     ([(2000, 100 + 50 * i) for i in range(8)], 128),  # 64 x 64
                                     ([(2000, 130), (3000, 70), (2500, 257)], 512)])   # 64 x 128
def test_grouped_small(bws, dev, sizes, N):
    probs = []
    for i, (M, K) in enumerate(sizes):
        B = torch.randn((K, N), device=dev).to(torch.bfloat16)
        probs.append((_mask(bws, dev, M, K, 0.1, i), B, torch.full((M, N), float("nan"), device=dev)))
    bws.spmm_batched(probs, "bf16")
    for A, B, C in probs:
        assert torch.equal(C, bws.spmm(A, B, "bf16"))
