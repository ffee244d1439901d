"""FP32 products of value masks around the K below which the plain tiles run:
the same bits as the value product's tile, which a grouped launch always takes."""
import pytest
import torch

from _helpers import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [1, 15, 16, 17, 31, 32, 33, 48, 49])
@pytest.mark.parametrize("M,N", [(1, 4), (70, 64), (300, 260), (1100, 4100), (129, 13)])
def test_same_bits(bws, dev, M, K, N):
    A = bws.Bitmap(to_dev(bws.gen_bitmap_iid(M + K, M, K, 0.4), dev), M, K)
    g = torch.Generator(device=dev).manual_seed(K)
    rp = bws.row_ptr(A)
    A = A.with_values(torch.randn(max(int(rp[-1]), 1), device=dev, generator=g), rp)
    B = torch.randn((K, N), device=dev, generator=g)
    C0 = torch.randn((M, N), device=dev, generator=g)
    C = bws.spmm(A, B)
    D = bws.unpack_bitmap(bws.Bitmap(A.words, M, K)).double()
    D[D != 0] = A.values[:int(rp[-1])].double()
    err = (C.double() - D @ B.double()).abs()
    assert bool((err <= (K + 2) * 2.0 ** -24 * (D.abs() @ B.double().abs())).all())
    E = bws.spmm(A, B, alpha=0.5, beta=-2.0, out=C0.clone())
    assert torch.equal(E, (0.5 * C.double() - 2.0 * C0.double()).float())
    if N % 4 == 0:  # (others leave the grouped launch)
        G = torch.empty_like(C)
        assert bws.spmm_batched([(A, B, G)]).launches[0]["kind"] == 1
        assert torch.equal(C, G)
