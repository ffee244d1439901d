"""FP32 products on the matrix cores where B holds values that its BF16 parts
cannot: infinities, NaN, values whose sums may overflow, tiny ones.  The
outputs over such columns are the vector-add kernels' bit for bit."""
import pytest
import torch

from _helpers import to_dev

pytestmark = pytest.mark.gpu

INF, NAN = float("inf"), float("nan")


def _same(x, y):
    """Equal bits, any NaN for a NaN."""
    return bool(((x == y) | (torch.isnan(x) & torch.isnan(y))).all())


def _streamed(bws, A, B, alpha, beta, C):
    """The product with room for the mask stream alone: the streamed kernel."""
    L, s = bws.lib(), A.struct()
    n = L.bws_spmm_workspace_size(bws.C.byref(s), B.shape[1], 0, None)
    ws = torch.empty(n, dtype=torch.uint8, device=B.device)
    assert L.bws_spmm(bws.C.byref(s), B.data_ptr(), 0, B.stride(0), B.shape[1], C.data_ptr(),
                      C.stride(0), alpha, beta, 0, None, ws.data_ptr(), n,
                      torch.cuda.current_stream().cuda_stream) == 0
    return C


@pytest.mark.parametrize("value", [INF, -INF, NAN, 2.0 ** 96, -3e38, 2.0 ** -101, 1e-45])
@pytest.mark.parametrize("M,K,N", [(4096, 200, 3076), (3841, 131, 3328)])
def test_routed_columns(bws, dev, M, K, N, value):
    """One such value in the first, an inner and the last 256 columns: those
    columns as the streamed kernel gives them, all others as without it."""
    A = bws.Bitmap(to_dev(bws.gen_bitmap_iid(M, M, K, 0.5), dev), M, K)
    g = torch.Generator(device=dev).manual_seed(K)
    B = torch.randn((K, N), device=dev, generator=g)
    C0 = torch.randn((M, N), device=dev, generator=g)
    plain = bws.spmm(A, B, alpha=0.5, beta=2.0, out=C0.clone())
    B[K - 1, 5] = B[0, 800] = B[K // 2, N - 1] = value
    C = bws.spmm(A, B, alpha=0.5, beta=2.0, out=C0.clone())
    S = _streamed(bws, A, B, 0.5, 2.0, C0.clone())
    held = torch.zeros(N, dtype=torch.bool, device=dev)
    held[:256] = held[768:1024] = held[(N - 1) // 256 * 256:] = True
    assert _same(C[:, held], S[:, held])
    assert torch.equal(C[:, ~held], plain[:, ~held]) and not torch.equal(plain[:, ~held], S[:, ~held])


@pytest.mark.parametrize("scale", [1e-25, 1e-35, 1e36])
def test_routed_scaled(bws, dev, scale):
    """A whole B out of the range, and zeros (which are in it) beside it."""
    M, K, N = 4096, 300, 3072
    A = bws.Bitmap(to_dev(bws.gen_bitmap_iid(7, M, K, 0.6), dev), M, K)
    B = torch.randn((K, N), device=dev) * scale
    B[::3, :256] = 0.0
    B[:, 512:768] = 0.0
    C = bws.spmm(A, B)
    S = _streamed(bws, A, B, 1.0, 0.0, torch.empty_like(C))
    assert bool((C[:, 512:768] == 0).all())
    wide = ((B != 0) & ((B.abs() < 2.0 ** -100) | (B.abs() >= 2.0 ** 96))).view(K, -1, 256).any(2).any(0)
    assert bool(wide.any())
    for i in torch.nonzero(wide).view(-1).tolist():
        assert _same(C[:, 256 * i:256 * i + 256], S[:, 256 * i:256 * i + 256])


# 8, 4 and 2 waves of the one-launch product; N past and off a lane's 8 columns
@pytest.mark.parametrize("M,K,N", [(300, 9000, 100), (3300, 4200, 301), (2048, 200, 1999)])
def test_direct_outputs(bws, dev, M, K, N):
    """Outputs over such values: the vector-add kernel's bits.  The others: the
    product's without them."""
    A = bws.Bitmap(to_dev(bws.gen_bitmap_iid(M, M, K, 0.1), dev), M, K)
    g = torch.Generator(device=dev).manual_seed(N)
    B = torch.randn((K, N), device=dev, generator=g)
    plain = bws.spmm(A, B)
    B[3, 1], B[K - 1, 2], B[5, N - 1], B[:, 8:16] = INF, NAN, -INF, 3e38
    B[:, 40:49] *= 1e-35
    B[:, 64] = 0.0
    B[0, 64] = 1e-42
    C0 = torch.randn((M, N), device=dev, generator=g)
    C = bws.spmm(A, B, alpha=-0.5, beta=0.25, out=C0.clone())
    V = bws.spmm(A, B, alpha=-0.5, beta=0.25, out=C0.clone(), plan=bws.make_plan(1))
    held = torch.zeros(N, dtype=torch.bool, device=dev)
    held[[1, 2, N - 1, 64]] = held[8:16] = held[40:49] = True
    assert _same(C[:, held], V[:, held])
    # (beta's term: one fused multiply-add)
    E = (0.25 * C0.double() - 0.5 * plain.double()).float()
    assert torch.equal(C[:, ~held], E[:, ~held])


def _us(f):
    best = 1e9
    for _ in range(5):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(4):
            f()
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b))
    return best


@pytest.mark.parametrize("M,K,N,p", [(1024, 1024, 1024, 0.1), (4096, 512, 3072, 0.3)])
def test_time_does_not_run_away(bws, dev, M, K, N, p):
    """An infinity in every column: within 10 times of ordinary values (4 and 2
    times measured; output by output it was 30 and more)."""
    A = bws.Bitmap(to_dev(bws.gen_bitmap_iid(1, M, K, p), dev), M, K)
    B = torch.randn((K, N), device=dev)
    C = torch.empty((M, N), device=dev)
    t0 = _us(lambda: bws.spmm(A, B, out=C))
    B[K // 2] = INF
    assert _us(lambda: bws.spmm(A, B, out=C)) <= 10 * t0
