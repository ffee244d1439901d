"""FP32 products of 0/1 masks on the matrix cores (B split exactly into three
BF16 parts): the one-launch kernel of small outputs and the dense side of the
density-routed product.  Sums of 3 K parts in any order, each addition rounded
or truncated to 24 bits, are within 3 K 2^-23 of sum |b|; sums of integers that
fit 24 bits are exact; a value that is not finite or too small for BF16 parts
acts on the rows that select it and on no other."""
import numpy as np
import pytest
import torch

from _helpers import to_dev

pytestmark = pytest.mark.gpu


def _mask(bws, dev, M, K, p, seed):
    W = bws.gen_bitmap_iid(seed, M, K, p)
    A = bws.Bitmap(to_dev(W, dev), M, K)
    return A, bws.unpack_bitmap(A).double()


def _check(C, D, B, K, alpha=1.0, beta=0.0, C0=None):
    R = alpha * (D @ B.double())
    S = abs(alpha) * (D @ B.double().abs())
    if C0 is not None:
        R += beta * C0.double()
        S += 2 * abs(beta) * C0.double().abs()
    bad = (C.double() - R).abs() > (3 * K + 4) * 2.0 ** -23 * S
    assert not bool(bad.any()), int(bad.sum())


# tile edges both ways, K below, at and past a step and a wave's share, N not a
# multiple of 4 and below 4, both wave counts (192 tiles and more)
DIRECT = [(1, 1, 1, 1.0), (64, 32, 64, 0.3), (63, 31, 61, 0.5), (65, 33, 67, 0.2),
          (130, 256, 2, 0.4), (70, 257, 5, 0.1), (128, 1000, 131, 0.05), (100, 40, 130, 0.9),
          (12300, 70, 64, 0.2), (64, 300, 12290, 0.1), (1500, 129, 1025, 0.02), (64, 5000, 3, 0.01),
          (2300, 100, 2301, 0.1), (4090, 40, 2306, 0.2)]  # rows off 16 bytes: up to 2304 tiles


@pytest.mark.parametrize("M,K,N,p", DIRECT)
def test_direct(bws, dev, M, K, N, p):
    A, D = _mask(bws, dev, M, K, p, M + K + N)
    g = torch.Generator(device=dev).manual_seed(N)
    B = torch.randn((K, N), device=dev, generator=g)
    _check(bws.spmm(A, B), D, B, K)
    # strided operands with 4-byte alignment only, alpha and beta
    Bs = torch.randn((K, N + 3), device=dev, generator=g)[:, 1:N + 1]
    Cs = torch.randn((M, N + 5), device=dev, generator=g)
    C0 = Cs.clone()
    bws.spmm(A, Bs, alpha=0.5, beta=-2.0, out=Cs[:, 3:3 + N])
    _check(Cs[:, 3:3 + N], D, Bs, K, 0.5, -2.0, C0[:, 3:3 + N])
    assert torch.equal(Cs[:, :3], C0[:, :3]) and torch.equal(Cs[:, 3 + N:], C0[:, 3 + N:])
    # integers: exact
    Bi = torch.randint(-1000, 1001, (K, N), device=dev, generator=g).float()
    assert torch.equal(bws.spmm(A, Bi).double(), D @ Bi.double())


# 192 and more tiles of 256 x 256: ragged rows, columns and K; the sparse side
# (5%) and both sides of the line of one bit in eight
@pytest.mark.parametrize("M,K,N", [(4096, 33, 3072), (4000, 200, 3000), (3841, 1, 3076)])
@pytest.mark.parametrize("p", [0.05, 0.11, 0.14, 0.5, 1.0])
def test_routed(bws, dev, M, K, N, p):
    A, D = _mask(bws, dev, M, K, p, M + K)
    g = torch.Generator(device=dev).manual_seed(K)
    B = torch.randn((K, N), device=dev, generator=g)
    _check(bws.spmm(A, B), D, B, K)
    C0 = torch.randn((M, N), device=dev, generator=g)
    _check(bws.spmm(A, B, alpha=2.0, beta=0.5, out=C0.clone()), D, B, K, 2.0, 0.5, C0)
    Bi = torch.randint(-1000, 1001, (K, N), device=dev, generator=g).float()
    assert torch.equal(bws.spmm(A, Bi).double(), D @ Bi.double())


def test_routed_small_workspace(bws, dev):
    """With the mask stream's workspace only, a dense mask takes the streamed
    kernel; both results are sums of the same integers."""
    M, K, N = 4096, 100, 3072
    A, D = _mask(bws, dev, M, K, 0.5, 3)
    B = torch.randint(-1000, 1001, (K, N), device=dev).float()
    s = A.struct()
    L = bws.lib()
    small = L.bws_spmm_workspace_size(bws.C.byref(s), N, 0, None)
    assert L.bws_spmm_best_workspace_size(bws.C.byref(s), N, 0, None) > small
    ws = torch.empty(small, dtype=torch.uint8, device=dev)
    out = torch.empty((M, N), device=dev)
    assert L.bws_spmm(bws.C.byref(s), B.data_ptr(), 0, N, N, out.data_ptr(), N, 1.0, 0.0, 0, None,
                      ws.data_ptr(), small, torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(out, bws.spmm(A, B)) and torch.equal(out.double(), D @ B.double())


@pytest.mark.parametrize("M,K,N", [(200, 150, 70), (4096, 90, 3072)])
def test_special_values(bws, dev, M, K, N):
    """Columns with an infinity, a NaN, sums that overflow, values below the
    range of the parts (FP32 subnormals among them) and a mixture of tiny and
    ordinary ones: every row is the FP32 sum of what it selects."""
    A, D = _mask(bws, dev, M, K, 0.3, 11)
    g = torch.Generator(device=dev).manual_seed(1)
    B = torch.randn((K, N), device=dev, generator=g)
    B[5, 3] = float("inf")
    B[6, 4] = float("nan")
    B[7, 5], B[8, 5] = float("inf"), float("-inf")
    B[:, 6] = 3e38
    B[:, 7] *= 1e-33
    B[:, 8] *= 1e-41
    B[::2, 9] *= 1e-36
    B[:, 10] = 0.0
    B[9, 10] = 1.4e-45
    B[:, 11] *= 1e36
    C = bws.spmm(A, B)
    # D is 0/1 and 0 * inf is not what a row that leaves the value out gets
    fin = torch.where(torch.isfinite(B), B, torch.zeros_like(B))
    R, S = D @ fin.double(), D @ fin.double().abs()
    for v in (float("inf"), float("-inf")):
        R = R + torch.where(D @ (B == v).double() > 0, torch.full_like(R, v), torch.zeros_like(R))
    R = torch.where(D @ torch.isnan(B).double() > 0, torch.full_like(R, float("nan")), R)
    R32 = R.float()
    assert torch.equal(torch.isnan(C), torch.isnan(R32))
    ok = torch.isfinite(R32)
    assert torch.equal(C[~ok & ~torch.isnan(C)], R32[~ok & ~torch.isnan(C)])
    err = (C.double() - R).abs()[ok]
    assert bool((err <= (3 * K + 4) * 2.0 ** -23 * S[ok] + 2.0 ** -149).all())


def test_direct_graph(bws, dev):
    """Captured with the routed product and replayed with eager work between."""
    A, _ = _mask(bws, dev, 300, 400, 0.1, 5)
    A2, _ = _mask(bws, dev, 4096, 64, 0.4, 6)
    B, B2 = torch.randn((400, 200), device=dev), torch.randn((64, 3072), device=dev)
    ref, ref2 = bws.spmm(A, B), bws.spmm(A2, B2)
    out, out2 = torch.empty_like(ref), torch.empty_like(ref2)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        with torch.cuda.graph(g, stream=s):
            bws.spmm(A, B, out=out)
            bws.spmm(A2, B2, out=out2)
    torch.cuda.current_stream().wait_stream(s)
    for _ in range(3):
        out.fill_(float("nan"))
        out2.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref) and torch.equal(out2, ref2)
        torch.randn(1 << 20, device=dev).cumsum(0)
        torch.cuda.synchronize()


@pytest.mark.parametrize("M,K,N", [(64, 40, 4), (1000, 300, 1100), (2048, 128, 2048), (2049, 65, 2052)])
def test_clustered_small_and_streamed(bws, dev, M, K, N):
    """The row-clustered product on both sides of 1024 tiles of 64 x 64."""
    A = bws.Bitmap(to_dev(bws.gen_bitmap_clustered(M, M, K, 16, 0.2, 0.02), dev), M, K)
    D = bws.unpack_bitmap(A).double()
    plan = bws.cluster_rows(A)
    B = torch.randn((K, N), device=dev)
    C0 = torch.randn((M, N), device=dev)
    _check(bws.spmm_clustered(A, plan, B, alpha=2.0, beta=0.5, out=C0.clone()), D, B, K, 2.0, 0.5, C0)
    Bi = torch.randint(-1000, 1001, (K, N), device=dev).float()
    assert torch.equal(bws.spmm_clustered(A, plan, Bi).double(), D @ Bi.double())
