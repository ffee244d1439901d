"""Split BF16 above 512 tiles of 64 x 64, where a workspace decides the kernel:
two passes over B's planes, or one that splits in registers.  (Smaller outputs
run in one launch either way.)"""
import pytest
import torch

from _helpers import to_dev

pytestmark = pytest.mark.gpu

# ragged M, K and N; N off 8: the planes' rows are padded (from K = 256, 512 and 1024)
SHAPES = [(2100, 97, 1352), (2100, 297, 1355), (1990, 1024, 1100), (4200, 257, 643), (4099, 513, 2501)]


def _product(bws, A, B, C, alpha, beta, ws):
    s = A.struct()
    assert bws.lib().bws_spmm(bws.C.byref(s), B.data_ptr(), 0, B.stride(0), B.shape[1], C.data_ptr(),
                              C.stride(0), alpha, beta, bws.PRECISION["bf16x2"], None,
                              None if ws is None else ws.data_ptr(), 0 if ws is None else ws.numel(),
                              torch.cuda.current_stream().cuda_stream) == 0
    return C


def _room(bws, A, N, dev):
    s = A.struct()
    n = bws.lib().bws_spmm_best_workspace_size(bws.C.byref(s), N, bws.PRECISION["bf16x2"], None)
    assert n > 0
    return torch.empty(n, dtype=torch.uint8, device=dev)


@pytest.mark.parametrize("M,K,N", SHAPES)
@pytest.mark.parametrize("alpha,beta,pad", [(1.0, 0.0, 0), (0.5, -2.0, 3)])
def test_two_forms(bws, dev, M, K, N, alpha, beta, pad):
    A = bws.Bitmap(to_dev(bws.gen_bitmap_iid(M, M, K, 0.4), dev), M, K)
    g = torch.Generator(device=dev).manual_seed(N)
    B = torch.randn((K, N + pad), device=dev, generator=g)[:, pad:]
    C0 = torch.randn((M, N + 2 * pad), device=dev, generator=g)
    D = bws.unpack_bitmap(A).double()
    c0 = C0[:, pad:pad + N].double()
    R = alpha * (D @ B.double()) + beta * c0
    S = abs(alpha) * (D @ B.double().abs()) + 2 * abs(beta) * c0.abs()
    out = []
    for ws in (_room(bws, A, N, dev), None):
        C = C0.clone()
        out.append(_product(bws, A, B, C[:, pad:pad + N], alpha, beta, ws))
        assert bool(((out[-1].double() - R).abs() <= 1e-5 * S).all())
        assert torch.equal(C[:, :pad], C0[:, :pad]) and torch.equal(C[:, pad + N:], C0[:, pad + N:])
    assert not torch.equal(out[0], out[1])  # two kernels


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_two_passes_round_once(bws, dev, M, K, N):
    """b = i + j/256, whole i in [129, 254], |j| <= 127: hi = i and lo = j/256, whose
    sums are exact; they meet in the second pass, in one rounding."""
    A = bws.Bitmap(to_dev(bws.gen_bitmap_iid(M + 1, M, K, 0.6), dev), M, K)
    g = torch.Generator(device=dev).manual_seed(K)
    B = (torch.randint(129, 255, (K, N), device=dev, generator=g).double()
         + torch.randint(-127, 128, (K, N), device=dev, generator=g).double() / 256)
    R = bws.unpack_bitmap(A).double() @ B
    C = torch.empty((M, N), device=dev)
    assert torch.equal(_product(bws, A, B.float(), C, 1.0, 0.0, _room(bws, A, N, dev)), R.float())


@pytest.mark.parametrize("M,K,N", [(1359, 128, 1351), (2000, 512, 1452), (6000, 640, 1004), (3000, 130, 1351),
                                   (4099, 300, 2501), (1000, 32, 1001)])
def test_short_k_in_registers(bws, dev, M, K, N):
    """N off 8 with a short K: no workspace is asked for, and one given is not used
    (the bits of the kernel that splits in registers, which a plan selects)."""
    A = bws.Bitmap(to_dev(bws.gen_bitmap_iid(M, M, K, 0.4), dev), M, K)
    B = torch.randn((K, N), device=dev, generator=torch.Generator(device=dev).manual_seed(N))
    s = A.struct()
    assert bws.lib().bws_spmm_best_workspace_size(bws.C.byref(s), N, bws.PRECISION["bf16x2"], None) == 0
    room = torch.empty(4 * K * (N + 8) + 4096, dtype=torch.uint8, device=dev)
    C = _product(bws, A, B, torch.empty((M, N), device=dev), 1.0, 0.0, room)
    assert torch.equal(C, bws.spmm(A, B, "bf16x2", plan=bws.make_plan(2)))
