"""Measured cases of the dense-contraction library: what its programs and
callers run, from the smallest polybench size to the largest benchmark
workload, every precision, operand order and entry point in use.

A case is a dict with a "kind":

- gemm:    C = alpha op(A) op(B) + beta C, one call (entry "gemm" or
           "gemm_noalloc"), any of the five precisions;
- syrk / syr2k: the triangle updates, mirrored (the polybench form) or not;
- covariance / correlation: column statistics, centring and the triangle
  product of an n x m data matrix;
- grouped: a batch of uneven problems, with a product chain beside them or
  without, as one call or as a replayed graph;
- chain:   the matmulchain product of `count` n x n matrices.

Inputs are uniform on [-1, 1) (the benchmark's distribution), sign x
lognormal(0, 2) for FP8 (its benchmark's), and columns with distinct means
and deviations for the statistics.  beta is 0 or 0.5, so that repeated passes
over one C stay bounded.
"""
import importlib.util
import math
import os
import sys

import torch

DEV = "cuda"
_mfx = None
_handle = None


def _lib():
    """The library's Python view, from the tree this file is run in."""
    global _mfx
    if _mfx is None:
        path = os.path.join(os.getcwd(), "sycl-bench_amd", "mfx.py")
        spec = importlib.util.spec_from_file_location("mfx", path)
        _mfx = importlib.util.module_from_spec(spec)
        sys.modules["mfx"] = _mfx
        spec.loader.exec_module(_mfx)
    return _mfx


def _h():
    """One handle for the process, as the benchmark programs keep."""
    global _handle
    if _handle is None:
        _handle = _lib().Handle(0)
    return _handle


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def _gemm(prec, m, n, k, ta=False, tb=False, beta=0.0, pad=0, entry="gemm"):
    return {"kind": "gemm", "entry": entry, "prec": prec, "m": m, "n": n, "k": k, "ta": ta, "tb": tb, "alpha": 1.5,
            "beta": beta, "pad": pad}


def _sym(kind, prec, n, k, uplo="lower", mirror=True, beta=0.5):
    return {"kind": kind, "prec": prec, "n": n, "k": k, "uplo": uplo, "mirror": mirror, "alpha": 1.5, "beta": beta}


def _stats(kind, prec, n, m):
    return {"kind": kind, "prec": prec, "n": n, "m": m}


def _grouped(prec, count, lo, hi, step, chain, chain_n, mode):
    return {"kind": "grouped", "prec": prec, "count": count, "lo": lo, "hi": hi, "step": step, "chain": chain,
            "chain_n": chain_n, "mode": mode}


def _chain(prec, count, n):
    return {"kind": "chain", "prec": prec, "count": count, "n": n}


def listed():
    return [
        # the smallest size of the polybench gemm in use: one tile, all launch latency
        dict(_gemm("fp32", 64, 64, 64, beta=0.5), name="gemm_fp32_64"),
        # polybench gemm at the suite's default --size=1024
        dict(_gemm("fp32", 1024, 1024, 1024, beta=0.5), name="gemm_fp32_1024"),
        # a ragged mid-size product with both operands transposed and padded
        # rows, through the entry point for callers that must not allocate
        dict(_gemm("split-bf16", 1000, 700, 1500, True, True, pad=4, entry="gemm_noalloc"), name="noalloc_split_ragged_tt"),
        # the headline benchmark
        dict(_gemm("split-bf16", 8192, 8192, 8192, beta=0.5), name="gemm_split_8192"),
        # the 2mm / 3mm size in single BF16, right operand stored transposed
        dict(_gemm("bf16", 4096, 4096, 4096, False, True), name="gemm_bf16_4096_nt"),
        # the FP8 benchmark, the largest call
        dict(_gemm("fp8-block", 16384, 16384, 16384), name="gemm_fp8_16384"),
        # two-term FP8 on an uneven mid-size product, left operand transposed
        dict(_gemm("fp8-block2", 1500, 1100, 2000, True, False), name="gemm_fp8x2_ragged_tn"),
        # polybench syrk at the default size: full square from one triangle
        dict(_sym("syrk", "fp32", 1024, 1024), name="syrk_fp32_1024"),
        # a larger symmetric update, one triangle only, sizes off the tile grid
        dict(_sym("syr2k", "split-bf16", 3000, 2500, mirror=False), name="syr2k_split_3000"),
        # correlation of many observations of a few hundred variables
        dict(_stats("correlation", "split-bf16", 20000, 500), name="correlation_split_20000x500"),
        # the batched benchmark: 512 uneven problems beside an 8-long chain, as a replayed graph
        dict(_grouped("split-bf16", 512, 64, 2048, 16, 8, 2048, "graph"), name="grouped_split_512_chain"),
        # runtime/matmulchain at the default size: (A B)(C D), one call
        dict(_chain("fp32", 4, 1024), name="chain_fp32_4x1024"),
    ]


def _log(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi, max(lo, int(round(v / step)) * step))


def _size(rng, lo, hi):
    """Log-uniform; half of them multiples of 16, the others as they fall (odd ones among them)."""
    return _log(rng, lo, hi, 16 if rng.random() < 0.5 else 1)


def draw(rng):
    kind = rng.choice(["gemm"] * 6 + ["syrk", "syr2k", "covariance", "correlation", "grouped", "chain"])
    if kind == "gemm":
        prec = rng.choice(["fp32", "split-bf16", "bf16", "fp8-block", "fp8-block2"])
        entry = "gemm"
        m, n, k = (_size(rng, 32, 8192) for _ in range(3))
        if prec in ("split-bf16", "bf16", "fp32") and rng.random() < 0.2:
            entry = "gemm_noalloc"  # its packed operands have to fit a fixed array
            m, n, k = (_size(rng, 32, 2048) for _ in range(3))
        return _gemm(prec, m, n, k, rng.random() < 0.5, rng.random() < 0.5, rng.choice([0.0, 0.5]), rng.choice([0, 0, 4]),
                     entry)
    if kind in ("syrk", "syr2k"):
        return _sym(kind, rng.choice(["fp32", "split-bf16", "bf16"]), _size(rng, 64, 6000), _size(rng, 64, 6000),
                    rng.choice(["lower", "upper"]), rng.random() < 0.5, rng.choice([0.0, 0.5]))
    if kind in ("covariance", "correlation"):
        return _stats(kind, rng.choice(["fp32", "split-bf16", "bf16"]), _size(rng, 64, 50000), _size(rng, 32, 2048))
    if kind == "grouped":
        lo = rng.choice([32, 64, 128])
        chain = rng.choice([0, 0, 4, 8])
        return _grouped(rng.choice(["fp32", "split-bf16", "bf16"]), _log(rng, 8, 256), lo, rng.choice([512, 1024, 2048]),
                        rng.choice([1, 16]), chain, _log(rng, 256, 2048, 16) if chain else 0,
                        rng.choice(["graph", "call"]))
    return _chain(rng.choice(["fp32", "split-bf16", "bf16"]), rng.choice([2, 4, 8]), _size(rng, 64, 2048))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _uniform(g, rows, cols, pad=0):
    """rows x cols on [-1, 1) in rows of cols + pad floats."""
    x = torch.rand((rows, cols + pad), generator=g, device=DEV).mul_(2.0).sub_(1.0)
    return x[:, :cols]


def _lognormal(g, rows, cols, pad=0):
    x = torch.randn((rows, cols + pad), generator=g, device=DEV).mul_(2.0).exp_()
    x.mul_(torch.randint(0, 2, x.shape, generator=g, device=DEV, dtype=torch.int8).mul_(2).sub_(1))
    return x[:, :cols]


def _gemm_inputs(case, seed):
    g = _gen(seed)
    make = _lognormal if case["prec"].startswith("fp8") else _uniform
    m, n, k, pad = case["m"], case["n"], case["k"], case["pad"]
    A = make(g, k, m, pad) if case["ta"] else make(g, m, k, pad)
    B = make(g, n, k, pad) if case["tb"] else make(g, k, n, pad)
    return A, B, _uniform(g, m, n, pad)


def _sym_inputs(case, seed):
    g = _gen(seed)
    A = _uniform(g, case["n"], case["k"])
    B = _uniform(g, case["n"], case["k"]) if case["kind"] == "syr2k" else None
    return A, B, _uniform(g, case["n"], case["n"])


def _data(case, seed):
    """n observations of m variables, each with a mean and a deviation of its own."""
    g = _gen(seed)
    n, m = case["n"], case["m"]
    mean = torch.rand((1, m), generator=g, device=DEV).mul_(4.0).sub_(2.0)
    dev = torch.rand((1, m), generator=g, device=DEV).add_(0.5)
    return torch.randn((n, m), generator=g, device=DEV).mul_(dev).add_(mean)


def _group_dims(case):
    """The batch's (m, n, k), log-uniform: the sizes belong to the case, not to the inputs' seed."""
    import random
    rng = random.Random(f"{case['count']}:{case['lo']}:{case['hi']}:{case['step']}")
    return [tuple(_log(rng, case["lo"], case["hi"], case["step"]) for _ in range(3)) for _ in range(case["count"])]


def _tree(count):
    """Balanced product tree over `count` inputs: (left, right) indices per product, inputs first, then products."""
    level, pairs, nxt = list(range(count)), [], count
    while len(level) > 1:
        up = []
        for i in range(0, len(level), 2):
            pairs.append((level[i], level[i + 1]))
            up.append(nxt)
            nxt += 1
        level = up
    return pairs


def _group_layout(case):
    """Offsets (in floats, 256-byte aligned) of every result in the batch's one result buffer, and its length."""
    shapes = [(m, n) for m, n, _ in _group_dims(case)]
    shapes += [(case["chain_n"], case["chain_n"])] * max(0, case["chain"] - 1)
    at, offs = 0, []
    for m, n in shapes:
        offs.append(at)
        at += (m * n + 63) // 64 * 64
    return shapes, offs, at


def _group_inputs(case, seed):
    g = _gen(seed)
    ops = [(_uniform(g, m, k), _uniform(g, k, n)) for m, n, k in _group_dims(case)]
    mats = [_uniform(g, case["chain_n"], case["chain_n"]) for _ in range(case["chain"])]
    return ops, mats


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "h": _h()}
    if kind == "gemm":
        s["A"], s["B"], s["C"] = _gemm_inputs(case, seed)
    elif kind in ("syrk", "syr2k"):
        s["A"], s["B"], s["C"] = _sym_inputs(case, seed)
    elif kind in ("covariance", "correlation"):
        n, m = case["n"], case["m"]
        s["data"] = _data(case, seed)
        s["mean"], s["sd"] = torch.empty(m, device=DEV), torch.empty(m, device=DEV)
        s["cen"], s["sym"] = torch.empty((n, m), device=DEV), torch.empty((m, m), device=DEV)
    elif kind == "chain":
        g = _gen(seed)
        n, count = case["n"], case["count"]
        s["mats"] = [_uniform(g, n, n) for _ in range(count)]
        s["scratch"] = [torch.empty((n, n), device=DEV) for _ in range(count - 2)]
        s["out"] = torch.empty((n, n), device=DEV)
    else:
        mfx = _lib()
        ops, mats = _group_inputs(case, seed)
        shapes, offs, total = _group_layout(case)
        flat = torch.zeros(total, device=DEV)
        outs = [flat[o:o + m * n].view(m, n) for (m, n), o in zip(shapes, offs)]
        base = len(ops)
        probs = [mfx.problem(a, b, c) for (a, b), c in zip(ops, outs)]
        deps = []
        every = mats + outs[base:]
        for i, (x, y) in enumerate(_tree(case["chain"]) if case["chain"] else []):
            probs.append(mfx.problem(every[x], every[y], outs[base + i]))
            deps += [(base + i, base + j - case["chain"]) for j in (x, y) if j >= case["chain"]]
        s.update(ops=ops, mats=mats, flat=flat, probs=probs, deps=deps)
        if case["mode"] == "graph":
            s["graph"] = s["h"].graph_create(probs, deps, prec=case["prec"])
    return s


def run(s):
    case, h = s["case"], s["h"]
    kind = case["kind"]
    if kind == "gemm":
        call = h.gemm_noalloc if case["entry"] == "gemm_noalloc" else h.gemm
        call(s["A"], s["B"], s["C"], alpha=case["alpha"], beta=case["beta"], prec=case["prec"], transA=case["ta"],
             transB=case["tb"])
        return s["C"]
    if kind in ("syrk", "syr2k"):
        mfx = _lib()
        opt = dict(alpha=case["alpha"], beta=case["beta"], prec=case["prec"], mirror=case["mirror"],
                   uplo=mfx.LOWER if case["uplo"] == "lower" else mfx.UPPER)
        if kind == "syrk":
            h.syrk(s["A"], s["C"], **opt)
        else:
            h.syr2k(s["A"], s["B"], s["C"], **opt)
        return s["C"]
    if kind == "covariance":
        h.covariance(s["data"], s["mean"], s["cen"], s["sym"], float(case["n"]), prec=case["prec"])
        return {"mean": s["mean"], "centered": s["cen"], "symmat": s["sym"]}
    if kind == "correlation":
        h.correlation(s["data"], s["mean"], s["sd"], s["cen"], s["sym"], float(case["n"]), 0.005, prec=case["prec"])
        return {"mean": s["mean"], "stddev": s["sd"], "centered": s["cen"], "symmat": s["sym"]}
    if kind == "chain":
        h.chain(s["mats"], s["scratch"], s["out"], prec=case["prec"])
        return s["out"]
    if case["mode"] == "graph":
        s["graph"].launch()
    else:
        h.grouped(s["probs"], s["deps"], prec=case["prec"])
    return s["flat"]


def exact(case, seed):
    kind = case["kind"]
    if kind == "gemm":
        A, B, C = _gemm_inputs(case, seed)
        A, B = A.double(), B.double()
        A, B = (A.T if case["ta"] else A), (B.T if case["tb"] else B)
        R = torch.matmul(A, B).mul_(case["alpha"])
        del A, B
        return R.add_(C.double(), alpha=case["beta"]) if case["beta"] else R
    if kind in ("syrk", "syr2k"):
        A, B, C = _sym_inputs(case, seed)
        A, C = A.double(), C.double()
        P = torch.matmul(A, A.T) if B is None else torch.matmul(A, B.double().T)
        P = P if B is None else P + P.T
        R = P.mul(case["alpha"]).add_(C, alpha=case["beta"])
        if case["mirror"]:
            return R
        keep = torch.ones_like(R, dtype=torch.bool)
        keep = keep.tril_() if case["uplo"] == "lower" else keep.triu_()
        return torch.where(keep, R, C)
    if kind in ("covariance", "correlation"):
        x = _data(case, seed).double()
        n = float(case["n"])
        mean = x.sum(0) / n
        c = x - mean
        if kind == "covariance":
            return {"mean": mean, "centered": c, "symmat": torch.matmul(c.T, c)}
        sd = (c.square().sum(0) / n).sqrt()
        sd = torch.where(sd <= 0.005, torch.ones_like(sd), sd)
        c = c / math.sqrt(n) / sd
        sym = torch.matmul(c.T, c)
        sym.fill_diagonal_(1.0)
        return {"mean": mean, "stddev": sd, "centered": c, "symmat": sym}
    if kind == "chain":
        g = _gen(seed)
        every = [_uniform(g, case["n"], case["n"]).double() for _ in range(case["count"])]
        for x, y in _tree(case["count"]):
            every.append(every[x] @ every[y])
        return every[-1]
    ops, mats = _group_inputs(case, seed)
    shapes, offs, total = _group_layout(case)
    flat = torch.zeros(total, device=DEV, dtype=torch.float64)
    outs = [a.double() @ b.double() for a, b in ops]
    every = [x.double() for x in mats]
    for x, y in _tree(case["chain"]) if case["chain"] else []:
        every.append(every[x] @ every[y])
    outs += every[case["chain"]:]
    for (m, n), o, r in zip(shapes, offs, outs):
        flat[o:o + m * n] = r.reshape(-1)
    return flat


def work(case):
    """Every input read once, every output written once (C read too when beta is not 0); a multiply-add is 2 operations."""
    kind = case["kind"]
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4 * (m * k + k * n + m * n * (2 if case["beta"] else 1)), "flops": 2 * m * n * k}
    if kind in ("syrk", "syr2k"):
        n, k, two = case["n"], case["k"], 2 if kind == "syr2k" else 1
        out = n * n if case["mirror"] else n * (n + 1) // 2
        return {"bytes": 4 * (two * n * k + out * (2 if case["beta"] else 1)), "flops": two * n * (n + 1) * k}
    if kind in ("covariance", "correlation"):
        n, m = case["n"], case["m"]
        per = 2 if kind == "covariance" else 6  # statistics and centring, per element
        return {"bytes": 4 * (2 * n * m + m * m + 2 * m), "flops": m * (m + 1) * n + per * n * m}
    if kind == "chain":
        n, c = case["n"], case["count"]
        return {"bytes": 4 * n * n * (c + 1), "flops": (c - 1) * 2 * n ** 3}
    b = sum(m * k + k * n + m * n for m, n, k in _group_dims(case))
    f = sum(2 * m * n * k for m, n, k in _group_dims(case))
    if case["chain"]:
        q, c = case["chain_n"], case["chain"]
        b += q * q * (2 * c - 1)
        f += (c - 1) * 2 * q ** 3
    return {"bytes": 4 * b, "flops": f}
