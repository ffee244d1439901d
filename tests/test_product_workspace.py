"""The workspace of a product in Python, on the host: what is asked for, and what
is taken where there is no memory for it."""
import pytest
import torch


def _struct(bws, M, K, values=False):
    return bws._Bitmap(M, K, bws.words_for(K), 4096, 4096 if values else None,
                       4096 if values else None)


# FP32 above 192 tiles of 256 x 256 (B's planes; else the mask stream), FP32 B
# padded to 16 bits, 16-bit B with rows off 16 bytes (else none)
CASES = [(4096, 4096, 4096, "fp32", torch.float32, True), (4096, 512, 4100, "fp32", torch.float32, True),
         (2000, 1000, 3001, "bf16", torch.float32, False), (2000, 1000, 3001, "bf16x2", torch.float32, False),
         (2000, 1000, 3001, "fp16", torch.float16, False)]


@pytest.mark.parametrize("M,K,N,precision,dtype,some", CASES)
def test_falls_back_without_memory(bws, monkeypatch, M, K, N, precision, dtype, some):
    s, B = _struct(bws, M, K), torch.empty((K, N), dtype=dtype, device="meta")
    monkeypatch.setattr(type(B), "data_ptr", lambda t: 4096, raising=False)
    L = bws.lib()
    args = (bws.C.byref(s), N, bws.PRECISION[precision], None)
    best, least = L.bws_spmm_best_workspace_size(*args), L.bws_spmm_workspace_size(*args)
    asked = []

    def short_of(limit):
        def alloc(n, device):
            asked.append(n)
            if n > limit:
                raise torch.OutOfMemoryError("no room")
            return n
        monkeypatch.setattr(bws, "_workspace", alloc)

    short_of(best)
    assert bws._product_workspace(s, B, precision, None) == best and asked == [best]
    short_of(best - 1)
    assert bws._product_workspace(s, B, precision, None) == (least if some else None)
    assert (least > 0) == some and least < best


def test_no_memory_at_all(bws, monkeypatch):
    """What was refused stays refused: the mask stream does not fit either."""
    def none(n, device):
        raise torch.OutOfMemoryError("no room")
    monkeypatch.setattr(bws, "_workspace", none)
    with pytest.raises(torch.OutOfMemoryError):
        bws._product_workspace(_struct(bws, 4096, 4096), torch.empty((4096, 4096), device="meta"),
                               "fp32", None)


def test_best_size(bws):
    """Without a plan: 0 for every output that runs without a workspace, else at
    least what bws_spmm_workspace_size reports; with a plan or values, just that."""
    L = bws.lib()
    for M in (64, 500, 2048, 4096):
        for K in (64, 1280, 2048):
            for N in (8, 300, 304, 1024, 4096):
                tiles = -(-M // 64) * -(-N // 64)
                for precision in ("fp32", "bf16", "fp16", "bf16x2"):
                    s, prec = _struct(bws, M, K), bws.PRECISION[precision]
                    args = (bws.C.byref(s), N, prec)
                    best, least = L.bws_spmm_best_workspace_size(*args, None), \
                        L.bws_spmm_workspace_size(*args, None)
                    if precision == "fp32":
                        none = -(-M // 256) * -(-N // 256) < 192
                    else:
                        none = tiles <= (512 if precision == "bf16x2" else 0 if K < 1280
                                         else 256 if K < 2048 else 512)
                    assert best == 0 if none else best >= least, (M, K, N, precision, best, least)
                    plan = bws.make_plan(1, 256, 16, 64)
                    v = _struct(bws, M, K, values=True)
                    for x, p in ((s, bws.C.byref(plan)), (v, None)):
                        assert L.bws_spmm_best_workspace_size(bws.C.byref(x), N, prec, p) == \
                            L.bws_spmm_workspace_size(bws.C.byref(x), N, prec, p)
