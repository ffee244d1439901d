"""A plan that names nothing selects the built-in defaults, as no plan does."""
import pytest
import torch

from _helpers import to_dev

pytestmark = pytest.mark.gpu

F32, B16, F16 = torch.float32, torch.bfloat16, torch.float16
# outputs of every route that is taken without a plan: one launch (FP32, 16 bits,
# split BF16), padded rows, the mask's density
CASES = [(1024, 1024, 512, "fp32", F32), (1024, 4096, 512, "bf16", B16), (500, 2000, 300, "fp16", F32),
         (500, 1000, 304, "bf16x2", F32), (2000, 300, 3001, "bf16", F32), (2000, 300, 3001, "fp16", F16),
         (4096, 256, 3072, "fp32", F32)]


@pytest.mark.parametrize("M,K,N,precision,dtype", CASES)
def test_same_bits(bws, dev, M, K, N, precision, dtype):
    A = bws.Bitmap(to_dev(bws.gen_bitmap_iid(M, M, K, 0.3), dev), M, K)
    B = torch.randn((K, N), device=dev, generator=torch.Generator(device=dev).manual_seed(N)).to(dtype)
    plan, s = bws.make_plan(), A.struct()
    assert torch.equal(bws.spmm(A, B, precision, plan=plan), bws.spmm(A, B, precision))
    for size in (bws.lib().bws_spmm_best_workspace_size, bws.lib().bws_spmm_workspace_size):
        assert size(bws.C.byref(s), N, bws.PRECISION[precision], bws.C.byref(plan)) == \
            size(bws.C.byref(s), N, bws.PRECISION[precision], None)
