"""Performance cases of the bit-wise SpMM library: the calls a program makes,
through the public entry points, over the range of sizes it makes them at.

A case is a dict of plain values.  Its ``kind`` says which calls make a pass:

* ``spmm``    C = A·B, A a 0/1 bitmap (a fixed sparsity pattern), in the case's
              precision: the forward of one sparse layer;
* ``rowplan`` the same FP32 product through the row-clustering plan a program
              builds once per mask;
* ``train``   one training step of a layer with a fixed mask and trainable
              values: C = A·B, dB = Aᵀ·dC, dvalues = (dC·Bᵀ) at the mask;
* ``grouped`` many uneven 0/1 problems (layers or experts), forward and dB, one
              grouped launch each way;
* ``mask``    what a program does with a new mask: pack, group its rows, bring
              it into transposed form and build the row-clustering plan.

Masks are drawn as a density (``p``) with either independent bits
(``mask="iid"``) or rows copied from ``protos`` prototypes of density ``p`` with
2% of the bits flipped (``mask="clustered"``).
"""
import math

import torch

import bitwise_spgemm_amd as bws

FLIP = 0.02
PROTOS = 64
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16,
          "bf16x2": torch.float32}


def _spmm(name, M, K, N, p, mask="iid", precision="fp32", b="normal"):
    return {"name": name, "kind": "spmm", "M": M, "K": K, "N": N, "p": p, "mask": mask,
            "precision": precision, "b": b}


def listed():
    return [
        # a small layer of a serving loop: the launches and the call itself count
        _spmm("fp32_small", 256, 512, 192, 0.05, "clustered"),
        # the 1024³ problem at 10%, the parity configuration
        _spmm("fp32_1024", 1024, 1024, 1024, 0.1),
        # sizes of nobody's tiles
        _spmm("fp32_ragged", 3001, 2053, 516, 0.05),
        # the headline workload: 4096³, 95% sparse, similar rows, the drop-in call
        _spmm("fp32_4096", 4096, 4096, 4096, 0.03125, "clustered"),
        # the dense end of the density sweep
        _spmm("fp32_4096_half", 4096, 4096, 4096, 0.5, "clustered"),
        # the headline workload with a mask that is kept: its plan is built once
        {"name": "rowplan_4096", "kind": "rowplan", "M": 4096, "K": 4096, "N": 4096,
         "p": 0.03125, "mask": "clustered", "b": "normal"},
        # 16-bit activations on the same mask
        _spmm("bf16_4096", 4096, 4096, 4096, 0.03125, "clustered", "bf16"),
        # 16-bit at an ordinary, uneven size
        _spmm("fp16_ragged", 1999, 3100, 1000, 0.1, "iid", "fp16"),
        # a training step with trainable values, FP32 and 16-bit
        {"name": "train_fp32", "kind": "train", "M": 4096, "K": 4096, "N": 2048, "p": 0.1,
         "mask": "iid", "precision": "fp32"},
        {"name": "train_bf16", "kind": "train", "M": 4096, "K": 4096, "N": 2048, "p": 0.1,
         "mask": "iid", "precision": "bf16"},
        # 32 uneven problems, M and K in [256, 8192], density 1-20%, forward and backward
        {"name": "grouped_bf16", "kind": "grouped", "count": 32, "N": 1024, "lo": 256, "hi": 8192,
         "step": 64, "sizes": 0},
        # a new 4096² mask
        {"name": "mask_4096", "kind": "mask", "M": 4096, "K": 4096, "p": 0.03125,
         "mask": "clustered", "tile_rows": 2048, "max_groups": 2},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["spmm", "spmm", "spmm", "spmm", "rowplan", "train", "grouped", "mask"])
    if kind == "grouped":
        return {"kind": kind, "count": rng.randint(4, 24), "N": rng.choice([128, 256, 512, 1000]),
                "lo": 256, "hi": rng.choice([2048, 4096]), "step": rng.choice([64, 1]),
                "sizes": rng.randrange(1 << 20)}
    M, K = _log(rng, 200, 4096), _log(rng, 200, 4096)
    mask = rng.choice(["iid", "clustered"])
    p = round(math.exp(rng.uniform(math.log(0.01), math.log(0.5))), 4)
    if kind == "mask":
        return {"kind": kind, "M": M, "K": K, "p": p, "mask": mask,
                "tile_rows": rng.choice([256, 1024, 2048]), "max_groups": rng.choice([2, 4])}
    # columns: a multiple of 64, of 4, or any number
    N = _log(rng, 100, 4096 if kind != "train" else 2048)
    N = max(64, N - N % rng.choice([64, 64, 4, 1]))
    if kind == "rowplan":
        return {"kind": kind, "M": M, "K": K, "N": N - N % 4, "p": p, "mask": "clustered",
                "b": rng.choice(["normal", "logu"])}
    if kind == "train":
        precision = rng.choice(["fp32", "bf16", "fp16"])
        return {"kind": kind, "M": M, "K": K, "N": N, "p": min(p, 0.2), "mask": mask,
                "precision": precision}
    case = _spmm("", M, K, N, p, mask, rng.choice(["fp32", "fp32", "bf16", "fp16", "bf16x2"]),
                 rng.choice(["normal", "normal", "logu"]))
    del case["name"]
    return case


def _density(p, mask):
    return p if mask == "iid" else p * (1 - FLIP) + (1 - p) * FLIP


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _mask(g, rows, cols, p, mask):
    """Dense boolean mask (rows x cols)."""
    if mask == "iid":
        return torch.rand((rows, cols), device="cuda", generator=g) < p
    proto = torch.rand((PROTOS, cols), device="cuda", generator=g) < p
    pick = torch.randint(PROTOS, (rows,), device="cuda", generator=g)
    flip = torch.rand((rows, cols), device="cuda", generator=g) < FLIP
    return proto[pick] ^ flip


def _mask_of(g, rows, cols, p, mask):
    """The same with exactly density * rows * cols set bits: the positions of
    the highest scores, where a clustered mask's bits come first."""
    n = int(round(_density(p, mask) * rows * cols))
    score = torch.rand((rows, cols), device="cuda", generator=g)
    if mask == "clustered":
        score += _mask(g, rows, cols, p, mask)
    top = score.view(-1).argsort(descending=True, stable=True)[:n]
    out = torch.zeros(rows * cols, dtype=torch.bool, device="cuda")
    out[top] = True
    return out.view(rows, cols)


def _dense(g, shape, dtype, b="normal"):
    if b == "normal":
        return torch.randn(shape, device="cuda", generator=g).to(dtype)
    # six decades of magnitudes with random signs
    mag = 10.0 ** (6.0 * torch.rand(shape, device="cuda", generator=g) - 3.0)
    sign = torch.rand(shape, device="cuda", generator=g) < 0.5
    return torch.where(sign, -mag, mag).to(dtype)


def _problem_sizes(case):
    """(M, K, density, mask kind) of every problem of a grouped case."""
    g = torch.Generator()
    g.manual_seed(case["sizes"])
    u = torch.rand((case["count"], 3), generator=g, dtype=torch.float64).tolist()
    lo, span, step = case["lo"], case["hi"] - case["lo"], case["step"]
    out = []
    for i, (a, b, c) in enumerate(u):
        out.append((lo + int(a * (span // step + 1)) * step, lo + int(b * (span // step + 1)) * step,
                    0.01 + 0.19 * c, "iid" if i % 2 == 0 else "clustered"))
    return out


def _inputs(case, seed):
    """The inputs of a case as plain tensors, from the seed alone."""
    g = _generator(seed)
    kind = case["kind"]
    if kind == "grouped":
        out = []
        for M, K, p, mask in _problem_sizes(case):
            out.append({"mask": _mask(g, M, K, p, mask),
                        "B": _dense(g, (K, case["N"]), torch.bfloat16),
                        "dC": _dense(g, (M, case["N"]), torch.bfloat16)})
        return out
    M, K = case["M"], case["K"]
    # trainable values: their number belongs to the layer, not to the draw
    mask = _mask_of if kind == "train" else _mask
    t = {"mask": mask(g, M, K, case["p"], case["mask"])}
    if kind in ("spmm", "rowplan"):
        t["B"] = _dense(g, (K, case["N"]), DTYPES[case.get("precision", "fp32")], case["b"])
    elif kind == "train":
        dt = DTYPES[case["precision"]]
        t["B"] = _dense(g, (K, case["N"]), dt)
        t["dC"] = _dense(g, (M, case["N"]), dt)
        t["values"] = 0.02 * _dense(g, (int(t["mask"].sum()),), torch.float32)
    else:
        t["D"] = torch.where(t["mask"], _dense(g, (M, K), torch.float32),
                             torch.zeros((), device="cuda"))
    return t


def prepare(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    state = {"case": case}
    if kind == "grouped":
        N = case["N"]
        fwd, bwd = [], []
        for p in t:
            A = bws.pack_bitmap(p["mask"].float())
            fwd.append((A, p["B"], torch.empty((A.rows, N), device="cuda")))
            bwd.append((bws.transpose(A), p["dC"], torch.empty((A.cols, N), device="cuda")))
        state["fwd"] = bws.Batch(fwd, "bf16")
        state["bwd"] = bws.Batch(bwd, "bf16")
        state["out"] = {"C": [x[2] for x in fwd], "dB": [x[2] for x in bwd]}
        return state
    if kind == "mask":
        state["D"] = t["D"]
        return state
    M, K, N = case["M"], case["K"], case["N"]
    A = bws.pack_bitmap(t["mask"].float())
    state.update(A=A, B=t["B"], C=torch.empty((M, N), device="cuda"))
    if kind == "rowplan":
        state["plan"] = bws.cluster_rows(A)
    elif kind == "train":
        state["A"] = A = A.with_values(t["values"], bws.row_ptr(A))
        AT, perm = bws.transpose_perm(A)
        nnz = t["values"].numel()
        state["AT"] = AT.with_values(torch.empty(nnz, device="cuda"), AT.row_ptr)
        state.update(perm=perm, dC=t["dC"], dB=torch.empty((K, N), device="cuda"),
                     dv=torch.empty(nnz, device="cuda"))
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "spmm":
        return bws.spmm(state["A"], state["B"], case["precision"], out=state["C"])
    if kind == "rowplan":
        return bws.spmm_clustered(state["A"], state["plan"], state["B"], out=state["C"])
    if kind == "train":
        A, AT, p = state["A"], state["AT"], case["precision"]
        C = bws.spmm(A, state["B"], p, out=state["C"])
        bws.gather(A.values, state["perm"], out=AT.values)
        dB = bws.spmm_tA(AT, state["dC"], p, out=state["dB"])
        dv = bws.sddmm(A, state["dC"], state["B"], p, out=state["dv"])
        return {"C": C, "dB": dB, "dvalues": dv}
    if kind == "grouped":
        state["fwd"].run()
        state["bwd"].run()
        return state["out"]
    A = bws.pack_bitmap(state["D"])
    groups = bws.group_rows(A, case["tile_rows"], case["max_groups"])
    AT = bws.transpose(A)
    plan = bws.cluster_rows(A)
    return {"words": A.words, "groups": groups, "transposed": AT.words,
            "slot_row": plan.slot_row, "chunk_mask": plan.chunk_mask}


def _spmm_work(M, K, N, density, esize, values=False):
    nnz = density * M * K
    nbytes = 4 * M * ((K + 31) // 32) + esize * K * N + 4 * M * N
    if values:
        nbytes += 4 * nnz + 8 * (M + 1)
    return nbytes, 2 * nnz * N


def work(case):
    kind = case["kind"]
    if kind == "grouped":
        nbytes = flops = 0
        for M, K, p, mask in _problem_sizes(case):
            for m, k in ((M, K), (K, M)):
                b, f = _spmm_work(m, k, case["N"], _density(p, mask), 2)
                nbytes += b
                flops += f
        return {"bytes": int(nbytes), "flops": int(flops)}
    M, K = case["M"], case["K"]
    density = _density(case["p"], case["mask"])
    if kind == "mask":
        words = 4 * M * ((K + 31) // 32)
        tiles = -(-M // case["tile_rows"]) * ((K + 31) // 32)
        groups = 4 * M * ((K + 31) // 32) + tiles * (4 * case["max_groups"] * 65 + 8 +
                                                     8 * case["tile_rows"])
        chunk_mask = 8 * -(-M // 16) * ((K + 31) // 32)
        return {"bytes": 4 * M * K + words + groups + 4 * K * ((M + 31) // 32) + 4 * M + chunk_mask,
                "flops": 0}
    N = case["N"]
    esize = DTYPES[case.get("precision", "fp32")].itemsize
    if kind == "train":
        nnz = density * M * K
        b0, f0 = _spmm_work(M, K, N, density, esize, True)
        b1, f1 = _spmm_work(K, M, N, density, esize, True)
        b2 = 4 * M * ((K + 31) // 32) + esize * (M + K) * N + 4 * nnz
        return {"bytes": int(b0 + b1 + b2 + 16 * nnz), "flops": int(f0 + f1 + 2 * nnz * N)}
    nbytes, flops = _spmm_work(M, K, N, density, esize)
    return {"bytes": int(nbytes), "flops": int(flops)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "mask":
        return None  # bitmaps, tables and copied values: no computed numbers
    t = _inputs(case, seed)
    if kind == "grouped":
        C, dB = [], []
        for p in t:
            D = p["mask"].double()
            C.append(D @ p["B"].double())
            dB.append(D.T.contiguous() @ p["dC"].double())
        return {"C": C, "dB": dB}
    D = t["mask"].double()
    B = t["B"].double()
    if kind != "train":
        return D @ B
    D[t["mask"]] = t["values"].double()
    dC = t["dC"].double()
    return {"C": D @ B, "dB": D.T.contiguous() @ dC,
            "dvalues": (dC @ B.T.contiguous())[t["mask"]]}
