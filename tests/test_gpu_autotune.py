"""The autotuner beside the built-in choice: a plan that it returns is never the
slower way to run a product."""
import pytest
import torch

from _helpers import make_problem, rel_err, to_dev

pytestmark = pytest.mark.gpu

B16 = torch.bfloat16


@pytest.fixture(autouse=True)
def _clean(bws):
    bws.lib().bws_autotune_clear()
    yield
    bws.lib().bws_autotune_clear()


# outputs that the built-in choice runs in one launch (2 to 4 times faster than
# any tile) or, with a workspace, by the mask's density
@pytest.mark.parametrize("M,K,N,precision,dtype", [(1024, 1024, 1024, "fp32", torch.float32),
                                                   (1024, 4096, 512, "bf16", B16),
                                                   (500, 2000, 304, "bf16x2", torch.float32),
                                                   (4096, 512, 3072, "fp32", torch.float32)])
def test_plan_runs_the_faster_one(bws, dev, M, K, N, precision, dtype):
    A = bws.Bitmap(to_dev(bws.gen_bitmap_iid(M, M, K, 0.3), dev), M, K)
    B = torch.randn((K, N), device=dev).to(dtype)
    plan, ms = bws.autotune(A, B, precision)
    assert plan.kernel in (1, 2) and plan.flags == 1 and ms > 0
    assert torch.equal(bws.spmm(A, B, precision, plan=plan), bws.spmm(A, B, precision))
    got = bws.autotune_lookup(M, K, N, A.nnz, precision)
    assert (got.kernel, got.rows_per_wg, got.flags) == (plan.kernel, plan.rows_per_wg, 1)


def test_tile_where_it_is_faster(bws, dev):
    """Short K: no built-in kernel but the tiles; the plan names one and runs it."""
    A = bws.Bitmap(to_dev(bws.gen_bitmap_iid(1, 512, 64, 0.05), dev), 512, 64)
    B = torch.randn((64, 512), device=dev)
    plan, _ = bws.autotune(A, B)
    assert plan.kernel == 1 and plan.rows_per_wg in (64, 128, 256)
    assert torch.equal(bws.spmm(A, B, plan=plan), bws.spmm(A, B))


def test_grouped_choice_is_the_batchs(bws, dev):
    """A small 16-bit batch: the cached tile leaves it the tiles of small outputs."""
    A = bws.Bitmap(to_dev(bws.gen_bitmap_iid(2, 1024, 4096, 0.1), dev), 1024, 4096)
    B, C = torch.randn((4096, 512), device=dev).to(B16), torch.empty((1024, 512), device=dev)
    plain = bws.spmm_batched([(A, B, C)], "bf16").launches[0]
    assert plain["rows"] < 128
    assert bws.autotune(A, B, "bf16", nnz=A.nnz)[0].flags == 1
    tuned = bws.spmm_batched([(A, B, C)], "bf16", nnz_hints=[A.nnz]).launches[0]
    assert (tuned["kind"], tuned["rows"], tuned["cols"]) == (plain["kind"], plain["rows"], plain["cols"])


def test_values_one_launch(oracle, bws, dev, tmp_path):
    """Value masks: tiles that differ in waves and stage alone are one kernel, and
    one grouped launch."""
    probs, refs = [], []
    for i in range(3):
        A, W, rp, v, B, Bd = make_problem(bws, oracle, dev, 300 << i, 200 << i, 256, 0.1, seed=i,
                                          values=True)
        probs.append((A, Bd, torch.empty((A.rows, 256), device=dev)))
        refs.append((W, B, rp, v))
        plan, _ = bws.autotune(A, Bd, nnz=int(rp[-1]))
        assert plan.waves_per_wg == 16 and plan.k_stage == (32 if plan.rows_per_wg == 64 else 64)
    path = tmp_path / "cache.txt"
    assert bws.lib().bws_autotune_save(str(path).encode()) == 0
    keys = [line.split()[:5] for line in path.read_text().splitlines() if not line.startswith("#")]
    assert len(keys) == 3
    other = [f"1 128 {w} {k} 0" for w, k in ((16, 64), (8, 64), (16, 32))]
    path.write_text("".join(" ".join(k) + " " + o + "\n" for k, o in zip(keys, other)))
    assert bws.lib().bws_autotune_load(str(path).encode()) == 0
    b = bws.spmm_batched(probs, nnz_hints=[int(r[2][-1]) for r in refs])
    assert [(x["rows"], x["count"]) for x in b.launches] == [(128, 3)]
    for (A, _, C), (W, B, rp, v) in zip(probs, refs):
        assert rel_err(oracle, C.cpu().numpy(), W, A.cols, B, rp, v)["max_rel_s"] <= 1e-5
