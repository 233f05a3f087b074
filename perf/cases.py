"""The work that users of this library have it do, as timed cases.

A case is a dict of plain values; `kind` names the entry point:
  block    block_gemm: many independent problems of one compiled shape, one call
  split    split_gemm: FP64 through FP16 / BF16 digits at sizes beyond the block shapes
  batched  BatchedPlan: problems of uneven size, the plan made once and executed many times
  spgemm   bsr_spgemm: block-sparse C = A * A, symbolic, fill and numeric phases
  spmm     bsr_spmm: a block-sparse A times a dense B
Distributions are those of the library's benchmark: U[-1, 1] for FP64 and batched
problems, signed log-uniform |x| in [1e-4, 1e4] for the split-precision paths, N(0, 1)
for FP16 / BF16 blocks and the sparse matrices.
"""
import math

import numpy as np
import torch

import kami_amd as K

DEV = "cuda"
PREC = {"f64": K.PREC_F64, "f16": K.PREC_F16_F32, "bf16": K.PREC_BF16_F32,
        "split_f16": K.PREC_F64_SPLIT_F16, "split_bf16": K.PREC_F64_SPLIT_BF16,
        "split_i8": K.PREC_F64_SPLIT_I8}
IN_DTYPE = {"f64": torch.float64, "f16": torch.float16, "bf16": torch.bfloat16,
            "split_f16": torch.float64, "split_bf16": torch.float64, "split_i8": torch.float64}
LOW = ("f16", "bf16")  # 2-byte inputs, FP32 results

# Shapes with a compiled block-GEMM instance, per precision.
SQUARE_F64 = [(16, 16, 16), (32, 32, 32), (64, 64, 64), (128, 128, 128), (64, 64, 512),
              (128, 128, 512)]
SQUARE_LOW = [(e, e, e) for e in (16, 32, 64, 128, 192, 208, 224, 256)]
LOWRANK = [(e, e, k) for e in (32, 64, 128, 192, 256) for k in (16, 32)]
SPLIT_BLOCK = [(64, 64, 64), (128, 128, 128)]


def listed():
    return [
        # the smallest call of a solver's inner loop: one wave of workgroups, all latency
        {"name": "block_f64_32_x64", "kind": "block", "prec": "f64", "m": 32, "n": 32, "k": 32,
         "count": 64, "layout": "nk"},
        # element matrices of an ordinary finite-element batch
        {"name": "block_f64_64_x1024", "kind": "block", "prec": "f64", "m": 64, "n": 64, "k": 64,
         "count": 1024, "layout": "nk"},
        # the benchmark's FP64 batch, native FP64 matrix instructions
        {"name": "block_f64_128_x4096", "kind": "block", "prec": "f64", "m": 128, "n": 128,
         "k": 128, "count": 4096, "layout": "nk"},
        # FP16 tiles of an ordinary mixed-precision batch
        {"name": "block_f16_128_x8192", "kind": "block", "prec": "f16", "m": 128, "n": 128,
         "k": 128, "count": 8192, "layout": "nk"},
        # the benchmark's FP64 batch through int8 digits
        {"name": "block_split_i8_128_x4096", "kind": "block", "prec": "split_i8", "m": 128,
         "n": 128, "k": 128, "count": 4096, "layout": "nk"},
        # one FP64 product of ordinary size through FP16 digits
        {"name": "split_f16_1024", "kind": "split", "prec": "split_f16", "m": 1024, "n": 1024,
         "k": 1024, "count": 1},
        # the benchmark's uneven batches: every M, N, K from 16 to 256
        {"name": "batched_f64_x20000", "kind": "batched", "prec": "f64", "count": 20000,
         "lo": 16, "hi": 256, "sizes": 3, "layout": "nk", "graph": True},
        {"name": "batched_f16_x20000", "kind": "batched", "prec": "f16", "count": 20000,
         "lo": 16, "hi": 256, "sizes": 3, "layout": "nk", "graph": True},
        # a short uneven batch in the K x N layout, as one step of a factorisation issues it
        {"name": "batched_bf16_kn_x500", "kind": "batched", "prec": "bf16", "count": 500,
         "lo": 16, "hi": 256, "sizes": 5, "layout": "kn", "graph": False},
        # the benchmark's sparse product, all phases
        {"name": "spgemm_f16_8192_2pct", "kind": "spgemm", "prec": "f16", "mb": 256, "bs": 32,
         "density": 0.02, "pattern": 4},
        # the benchmark's sparse-times-dense products
        {"name": "spmm_f16_8192_n256", "kind": "spmm", "prec": "f16", "mb": 256, "nb": 256,
         "bs": 32, "density": 0.02, "pattern": 4, "n": 256, "layout": "nk"},
        {"name": "spmm_f64_8192_n256", "kind": "spmm", "prec": "f64", "mb": 256, "nb": 256,
         "bs": 32, "density": 0.02, "pattern": 4, "n": 256, "layout": "nk"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# No drawn case moves more bytes or does more arithmetic than the largest listed ones.
MOST_BYTES, MOST_FLOPS = 1.5e9, 1.5e10


def draw(rng):
    """One more case: any entry point, precision and layout, sizes over the whole range."""
    kind = rng.choice(["block", "block", "split", "batched", "batched", "spgemm", "spmm"])
    if kind == "block":
        prec = rng.choice(["f64", "f64", "f16", "bf16", "split_i8", "split_f16"])
        m, n, k = rng.choice(SQUARE_F64 if prec == "f64" else SQUARE_LOW + LOWRANK if prec in LOW
                             else SPLIT_BLOCK)
        case = {"kind": kind, "prec": prec, "m": m, "n": n, "k": k, "count": 1,
                "layout": rng.choice(["nk", "nk", "kn"]) if prec in LOW + ("f64",) else "nk"}
    elif kind == "split":
        case = {"kind": kind, "prec": rng.choice(["split_f16", "split_f16", "split_bf16"]),
                "m": 64 * _log_int(rng, 1, 24), "n": 64 * _log_int(rng, 1, 24),
                "k": 32 * _log_int(rng, 1, 48), "count": 1}
    elif kind == "batched":
        lo, hi = rng.choice([(16, 64), (16, 256), (16, 256), (48, 400)])
        return {"kind": kind, "prec": rng.choice(["f64", "f64", "f16", "bf16"]),
                "count": _log_int(rng, 1, 20000 if hi < 400 else 3000), "lo": lo, "hi": hi,
                "sizes": rng.randrange(1 << 20), "layout": rng.choice(["nk", "nk", "kn"]),
                "graph": rng.random() < 0.5}
    elif kind == "spgemm":
        return {"kind": kind, "prec": rng.choice(["f64", "f16", "f16", "bf16"]),
                "mb": _log_int(rng, 8, 512), "bs": rng.choice([16, 32]),
                "density": round(math.exp(rng.uniform(math.log(0.005), math.log(0.08))), 4),
                "pattern": rng.randrange(1 << 20)}
    else:
        return {"kind": kind, "prec": rng.choice(["f64", "f64", "f16", "bf16"]),
                "mb": _log_int(rng, 8, 512), "nb": _log_int(rng, 8, 512),
                "bs": rng.choice([16, 32]),
                "density": round(math.exp(rng.uniform(math.log(0.005), math.log(0.2))), 4),
                "pattern": rng.randrange(1 << 20), "n": 16 * _log_int(rng, 1, 32), "layout": rng.choice(["nk", "nk", "kn"])}
    w = work(case)
    most = int(min(MOST_BYTES / w["bytes"], MOST_FLOPS / w["flops"]))
    if kind == "block":
        case["count"] = _log_int(rng, 1, max(1, min(most, 16384)))
    else:
        case["count"] = rng.choice([1, 1, 2, min(3, max(1, most))])
    return case


# ---------------------------------------------------------------- structure of a case

def _sizes(case):
    """M, N, K of every problem of a batch: log-uniform, multiples of 16."""
    rng = np.random.default_rng(case["sizes"])
    x = np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]), size=(case["count"], 3)))
    return np.clip(np.round(x / 16) * 16, 16, case["hi"]).astype(np.int64)


def _pattern(case):
    """Row pointers and ascending block columns of the sparse matrix: a random pattern."""
    rng = np.random.default_rng(case["pattern"])
    mb, nb = case["mb"], case.get("nb", case["mb"])
    nnzb = max(1, int(round(case["density"] * mb * nb)))
    at = np.sort(rng.choice(mb * nb, size=nnzb, replace=False))
    rp = np.zeros(mb + 1, np.int32)
    np.cumsum(np.bincount(at // nb, minlength=mb), out=rp[1:])
    return rp, (at % nb).astype(np.int32)


def _pairs(rp, ci):
    """(A block, B block, C row, C column) of every block product of A * A."""
    row = np.repeat(np.arange(len(rp) - 1), np.diff(rp))
    reps = rp[ci + 1] - rp[ci]
    a = np.repeat(np.arange(len(ci)), reps)
    start = np.cumsum(reps) - reps
    b = np.arange(len(a)) - np.repeat(start, reps) + rp[ci[a]]
    return a, b, row[a], ci[b]


def work(case):
    ei = 2 if case["prec"] in LOW else 8
    eo = 4 if case["prec"] in LOW else 8
    kind = case["kind"]
    if kind in ("block", "split"):
        m, n, k, c = case["m"], case["n"], case["k"], case["count"]
        return {"bytes": float(c) * (ei * (m * k + n * k) + eo * m * n), "flops": 2.0 * m * n * k * c}
    if kind == "batched":
        s = _sizes(case).astype(np.float64)
        m, n, k = s[:, 0], s[:, 1], s[:, 2]
        return {"bytes": float((ei * (m * k + n * k) + eo * m * n).sum()),
                "flops": float((2 * m * n * k).sum())}
    bs = case["bs"]
    if kind == "spgemm":
        rp, ci = _pattern(case)
        a, _, r, c = _pairs(rp, ci)
        out = len(np.unique(r.astype(np.int64) * case["mb"] + c))
        return {"bytes": float(len(ci) * (ei * bs * bs + 4) + out * (eo * bs * bs + 4) + 8 * len(rp)),
                "flops": 2.0 * max(1, len(a)) * bs ** 3}
    nnzb = max(1, int(round(case["density"] * case["mb"] * case["nb"])))
    return {"bytes": float(nnzb * (ei * bs * bs + 4) + ei * case["n"] * case["nb"] * bs +
                           eo * case["mb"] * bs * case["n"]),
            "flops": 2.0 * nnzb * bs * bs * case["n"]}


# ---------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000003 * int(seed) + 17)
    return g


def _normal(g, shape, prec):
    if prec in LOW:
        return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32).to(IN_DTYPE[prec])
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float64)


def _uniform(g, shape, prec):
    x = torch.rand(shape, generator=g, device=DEV, dtype=torch.float64 if prec not in LOW else torch.float32)
    return (x * 2 - 1).to(IN_DTYPE[prec])


def _log_uniform(g, shape):
    x = torch.rand(shape, generator=g, device=DEV, dtype=torch.float64).mul_(8).sub_(4)
    x = torch.pow(10.0, x)
    sign = torch.rand(shape, generator=g, device=DEV, dtype=torch.float32) < 0.5
    return torch.where(sign, -x, x)


def _dense(case, seed):
    """A and B of a block or split case."""
    g, c, prec = _gen(seed), case["count"], case["prec"]
    m, n, k = case["m"], case["n"], case["k"]
    bshape = (c, k, n) if case.get("layout") == "kn" else (c, n, k)
    if prec in LOW:
        return _normal(g, (c, m, k), prec), _normal(g, bshape, prec)
    if prec == "f64":
        return _uniform(g, (c, m, k), prec), _uniform(g, bshape, prec)
    return _log_uniform(g, (c, m, k)), _log_uniform(g, bshape)


def _batch(case, seed):
    """Flat operand buffers of a batch and each problem's view of A and B."""
    g, s = _gen(seed), _sizes(case)
    m, n, k = s[:, 0], s[:, 1], s[:, 2]
    a = _uniform(g, int((m * k).sum()), case["prec"])
    b = _uniform(g, int((n * k).sum()), case["prec"])
    views, oa, ob = [], 0, 0
    for mi, ni, ki in s.tolist():
        bv = b[ob:ob + ni * ki]
        views.append((a[oa:oa + mi * ki].view(mi, ki),
                      bv.view(ki, ni) if case["layout"] == "kn" else bv.view(ni, ki)))
        oa += mi * ki
        ob += ni * ki
    return s, views


def _sparse(case, seed):
    """Pattern and values of the block-sparse matrix, and the dense operand of an spmm."""
    g, bs = _gen(seed), case["bs"]
    nb = case.get("nb", case["mb"])
    rp, ci = _pattern(case)
    vals = _normal(g, (len(ci), bs, bs), case["prec"])
    if case["kind"] == "spgemm":
        return rp, ci, vals, None
    shape = (nb * bs, case["n"]) if case["layout"] == "kn" else (case["n"], nb * bs)
    return rp, ci, vals, _normal(g, shape, case["prec"])


def _bsr(case, rp, ci, vals):
    nb = case.get("nb", case["mb"])
    return K.BsrMatrix(case["mb"], nb, case["bs"], torch.from_numpy(rp).to(DEV),
                       torch.from_numpy(ci).to(DEV), vals)


def prepare(case, seed):
    kind, prec = case["kind"], case["prec"]
    out = torch.float32 if prec in LOW else torch.float64
    if kind in ("block", "split"):
        A, B = _dense(case, seed)
        C = torch.empty((case["count"], case["m"], case["n"]), dtype=out, device=DEV)
        return {"case": case, "A": A, "B": B, "C": C}
    if kind == "batched":
        s, views = _batch(case, seed)
        C = torch.empty(int((s[:, 0] * s[:, 1]).sum()), dtype=out, device=DEV)
        probs, oc = [], 0
        for (A, B), (m, n, _) in zip(views, s.tolist()):
            probs.append((A, B, C[oc:oc + m * n].view(m, n)))
            oc += m * n
        plan = K.BatchedPlan(probs, b_layout=case["layout"], use_graph=case["graph"])
        return {"case": case, "plan": plan, "C": C}
    rp, ci, vals, B = _sparse(case, seed)
    A = _bsr(case, rp, ci, vals)
    if kind == "spgemm":
        return {"case": case, "A": A}
    C = torch.empty((case["mb"] * case["bs"], case["n"]), dtype=out, device=DEV)
    return {"case": case, "A": A, "B": B, "C": C}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "block":
        return K.block_gemm(state["A"], state["B"], state["C"], precision=PREC[case["prec"]],
                            b_layout=case["layout"])
    if kind == "split":
        return K.split_gemm(state["A"], state["B"], state["C"], precision=PREC[case["prec"]])
    if kind == "batched":
        state["plan"].execute()
        return state["C"]
    if kind == "spgemm":
        c = K.bsr_spgemm(state["A"], state["A"])
        return c.rowptr, c.colidx, c.vals
    return K.bsr_spmm(state["A"], state["B"], state["C"], b_layout=case["layout"])


# ---------------------------------------------------------------- 64-bit results

def exact(case, seed):
    kind = case["kind"]
    if kind in ("block", "split"):
        A, B = _dense(case, seed)
        B = B.double()
        if case.get("layout") != "kn":
            B = B.transpose(1, 2).contiguous()
        return torch.bmm(A.double(), B)
    if kind == "batched":
        _, views = _batch(case, seed)
        return torch.cat([(A.double() @ (B.double() if case["layout"] == "kn" else B.double().t())).reshape(-1)
                          for A, B in views])
    rp, ci, vals, B = _sparse(case, seed)
    bs = case["bs"]
    if kind == "spgemm":
        a, b, r, c = _pairs(rp, ci)
        if not len(a):
            return None
        key = r.astype(np.int64) * case["mb"] + c
        out, at = np.unique(key, return_inverse=True)
        C = torch.zeros((len(out), bs, bs), dtype=torch.float64, device=DEV)
        step = 1 << 16
        for lo in range(0, len(a), step):
            ia, ib = (torch.from_numpy(np.ascontiguousarray(x[lo:lo + step])).to(DEV) for x in (a, b))
            C.index_add_(0, torch.from_numpy(at.reshape(-1)[lo:lo + step]).to(DEV),
                         torch.bmm(vals[ia].double(), vals[ib].double()))
        rowptr = np.zeros(case["mb"] + 1, np.int64)
        np.cumsum(np.bincount(out // case["mb"], minlength=case["mb"]), out=rowptr[1:])
        return rowptr.astype(np.int32), (out % case["mb"]).astype(np.int32), C
    dense = torch.zeros((case["mb"], case["nb"], bs, bs), dtype=torch.float64, device=DEV)
    row = np.repeat(np.arange(case["mb"]), np.diff(rp))
    dense[torch.from_numpy(row).to(DEV), torch.from_numpy(ci.astype(np.int64)).to(DEV)] = vals.double()
    dense = dense.permute(0, 2, 1, 3).reshape(case["mb"] * bs, case["nb"] * bs)
    B = B.double()
    return dense @ (B if case["layout"] == "kn" else B.t())
