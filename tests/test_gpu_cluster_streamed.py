"""The streamed row-clustered product, which runs above 1024 tiles of 64 x 64:
subtracting rows, strides, alpha and beta, empty rows, ragged edges.  (The
smaller outputs of test_gpu_cluster run in one launch from the bitmap.)"""
import numpy as np
import pytest
import torch

from _helpers import sampled_err, to_dev, to_host_u32

pytestmark = pytest.mark.gpu


def _streamed(bws, A, N, dev):
    """The product takes its masks from the plan: an empty plan gives zeros."""
    empty = bws.cluster_rows(bws.Bitmap(torch.zeros_like(A.words), A.rows, A.cols))
    return not bool(bws.spmm_clustered(A, empty, torch.ones((A.cols, N), device=dev)).any())


def _clustered(bws, dev, M, K, p, seed):
    W = bws.gen_bitmap_clustered(seed, M, K, 16, p, 0.02)
    return W, bws.Bitmap(to_dev(W, dev), M, K)


@pytest.mark.parametrize("M,K,N,p", [(4100, 700, 1060, 0.05), (2049, 65, 2116, 0.2), (16500, 33, 260, 0.3),
                                     (257, 1000, 13316, 0.1)])
def test_ragged(oracle, bws, dev, M, K, N, p):
    W, A = _clustered(bws, dev, M, K, p, M + N)
    B = bws.gen_f32(M + 1, (K, N), "normal", 0.0, 1.0)
    plan = bws.cluster_rows(A)
    assert _streamed(bws, A, N, dev)
    C = bws.spmm_clustered(A, plan, to_dev(B, dev))
    e = sampled_err(oracle, C, W, K, B, np.unique(np.r_[np.arange(0, M, 37), M - 1]))
    assert e["max_rel_s"] <= 1e-5, e


def test_many_subtracts(oracle, bws, dev, rng):
    """Nearly every slot subtracts in nearly every stage: the inline pair of
    subtract masks and the full table (three and more in a stage)."""
    M, K, N = 512, 1000, 8260
    D = ((rng.random(K) < 0.5)[None, :] & ~(rng.random((M, K)) < 0.2)) | (rng.random((M, K)) < 0.01)
    W = oracle.pack_bitmap(D.astype(np.float32))
    A = bws.Bitmap(to_dev(W, dev), M, K)
    B = bws.gen_f32(12, (K, N), "normal", 0.0, 1.0)
    plan = bws.cluster_rows(A)
    slot, cm = plan.slot_row.cpu().numpy().astype(np.int64), to_host_u32(plan.chunk_mask)
    assert ((slot & bws.SLOT_DELTA) != 0).mean() > 0.9
    most = 0
    for c in range(M // 16):
        flagged = np.zeros((K + 63) // 64, np.int64)
        for sr in slot[16 * c:16 * c + 16]:
            if sr < 0 or not (sr & bws.SLOT_DELTA):
                continue
            base = oracle.unpack_bitmap(cm[c, 1 if sr & bws.SLOT_BASE1 else 0][None, :], K)[0] != 0
            flagged += np.add.reduceat(base & ~D[sr & (bws.SLOT_BASE1 - 1)], np.arange(0, K, 64)) > 0
        most = max(most, int(flagged.max()))
    assert most >= 3 and _streamed(bws, A, N, dev)
    C = bws.spmm_clustered(A, plan, to_dev(B, dev))
    e = sampled_err(oracle, C, W, K, B, np.arange(0, M, 5))
    assert e["max_rel_s"] <= 1e-5, e


def test_strides_alpha_beta_empty_rows(oracle, bws, dev, rng):
    M, K, N = 2100, 200, 2052
    W, _ = _clustered(bws, dev, M, K, 0.2, 5)
    W[::3] = 0
    A = bws.Bitmap(to_dev(W, dev), M, K)
    Bw = bws.gen_f32(6, (K, N + 4), "normal", 0.0, 1.0)
    C0 = rng.standard_normal((M, N + 8)).astype(np.float32)
    Bd, Cd = to_dev(Bw, dev)[:, :N], to_dev(C0, dev)
    plan = bws.cluster_rows(A)
    assert _streamed(bws, A, N, dev)
    bws.spmm_clustered(A, plan, Bd, alpha=0.5, beta=-2.0, out=Cd[:, 4:4 + N])
    D = bws.unpack_bitmap(A).double()
    R, S = D @ Bd.double(), D @ Bd.double().abs()
    c0 = to_dev(C0, dev).double()
    err = (Cd[:, 4:4 + N].double() - (0.5 * R - 2.0 * c0[:, 4:4 + N])).abs()
    assert bool((err <= 1e-5 * (0.5 * S + 2.0 * c0[:, 4:4 + N].abs()) + 1e-6).all())
    assert torch.equal(Cd[:, :4].double(), c0[:, :4]) and torch.equal(Cd[:, 4 + N:].double(), c0[:, 4 + N:])
    assert bool((bws.spmm_clustered(A, plan, Bd)[::3] == 0).all())


def test_benchmark_mask(oracle, bws, dev):
    """64 prototypes, density 1/32, 2% flips: most rows are delta rows."""
    M = K = 4096
    N = 1088
    W = bws.gen_bitmap_clustered(0, M, K, 64, 0.03125, 0.02)
    A = bws.Bitmap(to_dev(W, dev), M, K)
    plan = bws.cluster_rows(A)
    assert ((plan.slot_row.cpu().numpy() & bws.SLOT_DELTA) != 0).mean() > 0.9
    assert _streamed(bws, A, N, dev)
    B = bws.gen_f32(1, (K, N), "normal", 0.0, 1.0)
    e = sampled_err(oracle, bws.spmm_clustered(A, plan, to_dev(B, dev)), W, K, B, np.arange(0, M, 11))
    assert e["max_rel_s"] <= 1e-5, e


def test_one_launch_special_values(bws, dev):
    """The smaller outputs: infinities, NaN and tiny values as bws_spmm has them."""
    M, K, N = 500, 300, 132
    _, A = _clustered(bws, dev, M, K, 0.2, 3)
    plan = bws.cluster_rows(A)
    B = torch.randn((K, N), device=dev)
    assert not _streamed(bws, A, N, dev)
    B[3, 1], B[5, 2], B[:, 8:16] = float("inf"), float("nan"), 3e38
    B[:, 40:50] *= 1e-35
    C, V = bws.spmm_clustered(A, plan, B), bws.spmm(A, B, plan=bws.make_plan(1))
    held = [1, 2] + list(range(8, 16)) + list(range(40, 50))
    assert bool(((C == V) | (torch.isnan(C) & torch.isnan(V)))[:, held].all())
