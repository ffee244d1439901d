"""The three-part split of FP32 values is exact: where an output selects one
value it is that value, all 24 bits of it, in every matrix-core kernel; and the
products stay closer to 64 bits than the vector adds however long K is."""
import pytest
import torch

from _helpers import to_dev

pytestmark = pytest.mark.gpu


def _values(g, K, N, dev):
    """Random 24-bit significands, exponents from 2^-90 to 2^90, both signs."""
    m = torch.randint(1 << 23, 1 << 24, (K, N), device=dev, generator=g).double()
    e = torch.randint(-90, 91, (K, N), device=dev, generator=g).double()
    s = torch.randint(0, 2, (K, N), device=dev, generator=g).double() * 2 - 1
    return (s * m * 2.0 ** (e - 23)).float()


# 8, 4 and 2 waves; rows off 16 bytes; a tail of K; a second chunk of words
@pytest.mark.parametrize("M,K,N", [(300, 200, 96), (129, 9001, 33), (3300, 4200, 301), (2048, 1000, 2048),
                                   (2000, 193, 2001), (5000, 2049, 1003)])
def test_one_value_one_launch(bws, dev, M, K, N):
    g = torch.Generator(device=dev).manual_seed(M)
    pick = torch.randint(K, (M,), device=dev, generator=g)
    A = bws.pack_bitmap(torch.zeros((M, K), device=dev).scatter_(1, pick[:, None], 1.0))
    B = _values(g, K, N, dev)
    assert torch.equal(bws.spmm(A, B), B[pick])


@pytest.mark.parametrize("M,K,N", [(4096, 131, 3076), (3900, 400, 3200)])
def test_one_value_planes(bws, dev, M, K, N):
    """A dense mask and a B of one nonzero row."""
    A = bws.Bitmap(to_dev(bws.gen_bitmap_iid(M, M, K, 0.5), dev), M, K)
    g = torch.Generator(device=dev).manual_seed(K)
    D = bws.unpack_bitmap(A)
    for k in (0, 31, 32, K - 1):
        B = torch.zeros((K, N), device=dev)
        B[k] = _values(g, 1, N, dev)[0]
        assert torch.equal(bws.spmm(A, B), torch.where(D[:, k:k + 1] != 0, B[k][None, :], 0.0))


@pytest.mark.parametrize("M,K,N,p", [(512, 1024, 192, 0.05), (512, 16384, 192, 0.5), (512, 65536, 192, 0.05),
                                     (512, 65536, 191, 0.5), (3300, 32768, 301, 0.01),
                                     (4096, 16384, 3072, 0.3)])
@pytest.mark.parametrize("kind", ["positive", "decades", "normal"])
def test_closer_than_vector_adds(bws, dev, M, K, N, p, kind):
    """Values of one sign, where the matrix unit's truncated additions all err the
    same way, over six decades, and of both signs."""
    A = bws.Bitmap(to_dev(bws.gen_bitmap_iid(M + K, M, K, p), dev), M, K)
    g = torch.Generator(device=dev).manual_seed(N)
    u = torch.rand((K, N), device=dev, generator=g)
    B = u if kind == "positive" else 10.0 ** (6 * u - 3) if kind == "decades" else \
        torch.randn((K, N), device=dev, generator=g)
    rows = slice(0, 256)
    R = bws.unpack_bitmap(A)[rows].double() @ B.double()
    err = [float((C[rows].double() - R).norm() / R.norm())
           for C in (bws.spmm(A, B), bws.spmm(A, B, plan=bws.make_plan(1, 256, 16, 64)))]
    assert err[0] <= err[1], err
