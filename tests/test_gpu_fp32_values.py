"""FP32 products of value-carrying bitmaps: the tile kernel at the edges of its
row blocks, column blocks and K stages, B rows with and without 16-byte
alignment, masks from empty to full.  A chain of n fused multiply-adds is within
n 2^-24 / (1 - n 2^-24) of sum |v b|; alpha and beta add a rounding each."""
import numpy as np
import pytest
import torch

from _helpers import to_dev

pytestmark = pytest.mark.gpu


def _problem(bws, dev, M, K, N, p, seed):
    W = bws.gen_bitmap_iid(seed, M, K, p)
    A = bws.Bitmap(to_dev(W, dev), M, K)
    g = torch.Generator(device=dev).manual_seed(seed)
    D = bws.unpack_bitmap(A).double()
    v = torch.randn(int(D.sum().item()), device=dev, generator=g)
    D[D != 0] = v.double()  # row-major order of the set bits
    return A.with_values(v, bws.row_ptr(A)), D, torch.randn((K, N), device=dev, generator=g), g


def _check(C, D, B, alpha=1.0, beta=0.0, C0=None):
    R = alpha * (D @ B.double())
    S = abs(alpha) * (D.abs() @ B.double().abs())
    n = (D != 0).sum(1, keepdim=True).double() + 4
    if C0 is not None:
        R += beta * C0.double()
        S += 2 * abs(beta) * C0.double().abs()
    bad = (C.double() - R).abs() > n * 2.0 ** -23 * S
    assert not bool(bad.any()), int(bad.sum())


SHAPES = [(1, 1, 1, 1.0), (3, 31, 4, 0.5), (64, 64, 256, 0.1), (65, 65, 257, 0.3),
          (63, 63, 255, 0.02), (129, 128, 260, 0.01), (257, 200, 512, 0.05), (300, 1000, 2, 0.2),
          (100, 4097, 70, 0.003), (257, 129, 515, 1.0), (70, 300, 5, 0.0)]


@pytest.mark.parametrize("rows", [0, 64, 128, 256])
@pytest.mark.parametrize("M,K,N,p", SHAPES)
def test_values(bws, dev, M, K, N, p, rows):
    A, D, B, g = _problem(bws, dev, M, K, N, p, M + K + N)
    plan = bws.make_plan(kernel=1, rows_per_wg=rows) if rows else None
    _check(bws.spmm(A, B, plan=plan), D, B)
    # strided operands with 4-byte alignment only, alpha and beta
    Bs = torch.randn((K, N + 3), device=dev, generator=g)[:, 1:N + 1]
    Cs = torch.randn((M, N + 5), device=dev, generator=g)
    C0 = Cs.clone()
    bws.spmm(A, Bs, alpha=0.5, beta=-2.0, out=Cs[:, 3:3 + N], plan=plan)
    _check(Cs[:, 3:3 + N], D, Bs, 0.5, -2.0, C0[:, 3:3 + N])
    assert torch.equal(Cs[:, :3], C0[:, :3]) and torch.equal(Cs[:, 3 + N:], C0[:, 3 + N:])


@pytest.mark.parametrize("rows", [0, 64, 128, 256])
def test_not_finite(bws, dev, rows):
    """A row of B or a value that is not finite acts on the rows that select it."""
    A, D, B, _ = _problem(bws, dev, 200, 150, 64, 0.05, 9)
    B[7, 3], B[60, 5], B[149, 9] = float("inf"), float("nan"), float("-inf")
    A.values[11], A.values[40] = float("inf"), float("nan")
    plan = bws.make_plan(kernel=1, rows_per_wg=rows) if rows else None
    C = bws.spmm(A, B, plan=plan)
    used = D != 0
    vals = torch.zeros_like(D)
    vals[used] = A.values.double()
    bad_v = ~torch.isfinite(vals).all(1, keepdim=True)
    bad_b = (used.double() @ (~torch.isfinite(B)).double()) > 0
    assert torch.equal(~torch.isfinite(C), bad_v | bad_b)


def test_batch(bws, dev):
    """One grouped launch over problems of different shapes."""
    parts = [_problem(bws, dev, M, K, 256, p, i) for i, (M, K, p) in
             enumerate([(300, 200, 0.1), (64, 65, 0.5), (1000, 500, 0.01), (7, 300, 1.0)])]
    outs = [torch.empty((x[0].rows, 256), device=dev) for x in parts]
    bws.spmm_batched([(x[0], x[2], C) for x, C in zip(parts, outs)])
    for (A, D, B, _), C in zip(parts, outs):
        _check(C, D, B)
