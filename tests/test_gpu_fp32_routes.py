"""Short products of 0/1 masks at FP32 that the vector-add kernels finish first:
they take those, so they give those kernels' bits (sums in ascending k; the
matrix cores sum in another order and differ in some)."""
import pytest
import torch

from _helpers import to_dev

pytestmark = pytest.mark.gpu


def _operands(bws, dev, M, K, N, p):
    A = bws.Bitmap(to_dev(bws.gen_bitmap_iid(M + N, M, K, p), dev), M, K)
    return A, torch.randn((K, N), device=dev, generator=torch.Generator(device=dev).manual_seed(K))


# 16-byte rows below K = 160; others below 192 where there are more than 256 tiles
@pytest.mark.parametrize("M,K,N", [(256, 128, 256), (1024, 159, 1024), (500, 130, 64), (16384, 128, 65),
                                   (2000, 191, 2001), (32768, 128, 33)])
def test_one_launch_short_k(bws, dev, M, K, N):
    A, B = _operands(bws, dev, M, K, N, 0.3)
    assert torch.equal(bws.spmm(A, B), bws.spmm(A, B, plan=bws.make_plan(1)))


@pytest.mark.parametrize("M,K,N", [(256, 160, 256), (1000, 128, 1001), (2000, 192, 2001)])
def test_one_launch_from_there(bws, dev, M, K, N):
    A, B = _operands(bws, dev, M, K, N, 0.3)
    assert not torch.equal(bws.spmm(A, B), bws.spmm(A, B, plan=bws.make_plan(1)))


@pytest.mark.parametrize("M,K,N,streamed", [(2048, 64, 2048, True), (4096, 191, 1024, True),
                                            (1500, 16, 2048, True), (2048, 192, 2048, False),
                                            (1024, 64, 2048, False)])
def test_clustered_short_k(bws, dev, M, K, N, streamed):
    """Above 512 tiles the streamed kernel runs below K = 192: it takes the masks
    from the plan (an empty mask's plan gives zeros), the one-launch product from A."""
    A, B = _operands(bws, dev, M, K, N, 0.3)
    empty = bws.cluster_rows(bws.Bitmap(torch.zeros_like(A.words), M, K))
    C = bws.spmm_clustered(A, empty, B)
    assert bool((C == 0).all()) == streamed
    ref = bws.unpack_bitmap(A).double() @ B.double()
    bound = 1e-5 * (bws.unpack_bitmap(A).double() @ B.double().abs())
    assert bool(((bws.spmm_clustered(A, bws.cluster_rows(A), B).double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("M,K,N,streamed", [(4096, 32, 4096, True), (3072, 95, 4096, True),
                                            (3072, 96, 4096, False)])
def test_routed_short_k(bws, dev, M, K, N, streamed):
    """A dense mask of a large output: below K = 96 the streamed kernel's bits (its
    sums are the vector-add kernel's), and a workspace for the mask stream alone."""
    A, B = _operands(bws, dev, M, K, N, 0.5)
    assert torch.equal(bws.spmm(A, B), bws.spmm(A, B, plan=bws.make_plan(1))) == streamed
    L, s = bws.lib(), A.struct()
    sizes = [f(bws.C.byref(s), N, 0, None) for f in (L.bws_spmm_workspace_size,
                                                     L.bws_spmm_best_workspace_size)]
    assert (sizes[0] == sizes[1]) == streamed
