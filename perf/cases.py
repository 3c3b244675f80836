"""Performance cases of kraken_amd: the calls a tensor-parallel program makes, through the public functions.

One rank's part of the work is measured, as everywhere in this package: the other ranks' buffers are slices of one
tensor or separate tensors on the same GPU.  Four families of calls, each over the range of sizes it is used with:

* rows       reduce + bias + RMSNorm behind a row-parallel layer, and the stand-alone RMSNorm: one token up to a
             long prefill, model widths from 1024 to 16384;
* reduce     the plain all-reduce and its two-shot share, with and without a bias: messages from a few KiB to 32 MiB;
* gemm       GEMM + all-reduce and GEMM + reduce-scatter, a few decode rows up to a long prefill; bf16 operands, or
             fp32 operands (what the all-reduce form is called with when activations are kept in fp32);
* gather     all-gather + GEMM on bf16 or fp8 shards, gathered beforehand or copied while the product runs.

W is the number of ranks (8 on a full node).  Activations and partial sums are N(0, 1), bf16 weights N(0, 0.02), fp8
weights N(0, 0.25) (scaled into the format's range), biases N(0, 0.02), norm weights 1 + N(0, 0.02).
"""
import math

import torch

from kraken_amd import comm, fused

BF16, F32, FP8 = torch.bfloat16, torch.float32, torch.float8_e4m3fn

MAX_BYTES = 5.6e8      # what a drawn call may read and write: no more than the largest listed one
MAX_FLOPS = 9.0e11     # and compute, in bf16 terms: likewise


# ---- the listed cases ---------------------------------------------------------------------------
def listed():
    return [
        # one decode step's 16 tokens through a row-parallel layer of width 8192: the smallest call, all latency
        {"name": "rows_decode", "op": "rms", "W": 8, "rows": 16, "D": 8192, "bias": "vector", "x": False},
        # a chunk of 512 tokens at width 5120, called as the reference's benchmark does: this rank's input as a
        # tensor of its own, a bias of the input's shape
        {"name": "rows_chunk", "op": "rms", "W": 8, "rows": 512, "D": 5120, "bias": "full", "x": True},
        # the plain one-shot all-reduce of a 4096 x 4096 message: HBM streaming
        {"name": "reduce_32mib", "op": "reduce", "W": 8, "rows": 4096, "D": 4096, "bias": "none", "share": "all"},
        # this rank's share of a two-shot all-reduce + bias, interleaved ownership, an odd number of rows
        {"name": "two_shot_share", "op": "reduce", "W": 8, "rows": 2047, "D": 5120, "bias": "full", "share": "striped"},
        # 16 decode tokens through the row-parallel down-projection (K = 3584 of 28672) and its all-reduce
        {"name": "gemm_ar_decode", "op": "ar", "W": 8, "M": 16, "N": 8192, "K": 3584, "b_t": True, "dtype": "bf16",
         "out": "bf16", "bias": False},
        # 4096 prefill tokens through a row-parallel output projection (K = 1024 of 8192), all-reduce and bias
        {"name": "gemm_ar_prefill", "op": "ar", "W": 8, "M": 4096, "N": 8192, "K": 1024, "b_t": False, "dtype": "bf16",
         "out": "bf16", "bias": True},
        # fp32 operands and result (the all-reduce form's default result), a ragged number of tokens
        {"name": "gemm_ar_fp32", "op": "ar", "W": 4, "M": 1000, "N": 4096, "K": 2048, "b_t": False, "dtype": "fp32",
         "out": "fp32", "bias": False},
        # a chunk of 512 tokens, GEMM + reduce-scatter, in the middle of the reference's sweep of shapes
        {"name": "gemm_rs_chunk", "op": "rs", "W": 8, "M": 512, "N": 6656, "K": 8192, "b_t": True, "dtype": "bf16"},
        # 8192 prefill tokens through the row-parallel down-projection and its reduce-scatter
        {"name": "gemm_rs_prefill", "op": "rs", "W": 8, "M": 8192, "N": 8192, "K": 3584, "b_t": False, "dtype": "bf16"},
        # the copy-engine form of the reduce-scatter at its reference shape, every band sent out: the largest call
        {"name": "gemm_rs_copy", "op": "rs_ce", "W": 8, "M": 8192, "N": 4096, "K": 14336, "b_t": True, "dtype": "bf16"},
        # 8192 prefill tokens, column-parallel product while the eight shards arrive
        {"name": "gather_overlap", "op": "ag", "W": 8, "m": 1024, "N": 3584, "K": 8192, "dtype": "bf16", "gather": True},
        # fp8 shards of 500 tokens each (no multiple of a tile), already gathered
        {"name": "gather_fp8", "op": "ag", "W": 8, "m": 500, "N": 6656, "K": 4096, "dtype": "fp8", "gather": False},
    ]


# ---- drawn cases --------------------------------------------------------------------------------
def _spread(rng, lo, hi, step=1):
    """A multiple of ``step`` in [lo, hi], spread evenly over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi // step * step, max(-(-lo // step) * step, int(round(v / step)) * step))


def _ranks(rng):
    return rng.choice((2, 4, 8, 8, 8, 3, 6, 16))


def draw(rng):
    op = rng.choice(("rms", "rms", "norm", "reduce", "reduce", "ar", "ar", "rs", "rs", "rs_ce", "ag", "ag"))
    if op in ("rms", "norm", "reduce"):
        c = {"op": op, "W": 1 if op == "norm" else _ranks(rng), "rows": _spread(rng, 1, 16384),
             "D": _spread(rng, 1024, 16384, 64)}
        if op == "rms":
            c.update(bias=rng.choice(("vector", "full", "none")), x=rng.random() < 0.5)
        elif op == "reduce":
            c.update(bias=rng.choice(("none", "none", "vector", "full")), share=rng.choice(("all", "all", "rows", "striped")))
            if c["share"] == "rows":       # whole rows for every rank
                c["rows"] = -(-c["rows"] // c["W"]) * c["W"]
            if c["share"] == "striped":    # ownership in blocks needs a block every rank count divides, a full bias
                c["W"] = rng.choice((2, 4, 8))
                c["bias"] = rng.choice(("none", "full"))
        step = c["W"] if c.get("share") == "rows" else 1
        while work(c)["bytes"] > MAX_BYTES:
            c["rows"] = max(step, c["rows"] // 2 // step * step)
        return c
    # products: N and K are model dimensions (multiples of 64, now and then only of 16), rows are tokens
    dim = 64 if rng.random() < 0.8 else 16
    c = {"op": op, "W": rng.choice((2, 4, 8, 8))}
    if op == "ag":
        c.update(m=_spread(rng, 1, 1024), N=_spread(rng, 1024, 8192, dim), K=_spread(rng, 1024, 16384, dim),
                 dtype=rng.choice(("bf16", "bf16", "fp8")), gather=rng.random() < 0.5)
        rows = "m"
    else:
        c.update(M=_spread(rng, 1, 8192), N=_spread(rng, 1024, 8192, dim), K=_spread(rng, 512, 16384, dim),
                 b_t=rng.random() < 0.5, dtype="fp32" if op == "ar" and rng.random() < 0.4 else "bf16")
        if op == "ar":
            c.update(out=rng.choice(("bf16", "fp32")) if c["dtype"] == "bf16" else "fp32", bias=rng.random() < 0.5)
        rows = "M"
    step = 1 if op in ("ar", "ag") else c["W"]
    c[rows] = -(-c[rows] // step) * step
    cost = 3.0 if c["dtype"] == "fp32" else 1.0
    while cost * work(c)["flops"] > MAX_FLOPS or work(c)["bytes"] > MAX_BYTES:
        c[rows] = max(step, c[rows] // 2 // step * step)
    return c


# ---- what a program has in hand -----------------------------------------------------------------
def prepare(case, seed):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev)
    g.manual_seed(seed)

    def randn(*shape, std=1.0, mean=0.0, dtype=BF16):
        t = torch.randn(shape, generator=g, device=dev, dtype=F32)
        if std != 1.0:
            t.mul_(std)
        if mean != 0.0:
            t.add_(mean)
        return t.to(dtype)

    op, W = case["op"], case["W"]
    s = {"op": op, "case": case}
    if op in ("rms", "norm", "reduce"):
        rows, D = case["rows"], case["D"]
        if op == "norm":
            return dict(s, x=randn(rows, D), w=randn(D, std=0.02, mean=1.0))
        s["stack"] = randn(W, rows, D)
        s["bias"] = {"none": lambda: None, "vector": lambda: randn(D, std=0.02),
                     "full": lambda: randn(rows, D, std=0.02)}[case["bias"]]()
        if op == "rms":
            s["x"] = randn(rows, D) if case["x"] else None
            s["w"] = randn(D, std=0.02, mean=1.0)
            s["y"] = torch.empty(rows, D, dtype=BF16, device=dev)
        elif case["bias"] != "none":
            n = rows * D
            share = {"all": n, "rows": n // W, "striped": _striped_numel(n, W, RANK, STRIPE)}[case["share"]]
            s["out"] = torch.empty(share, dtype=BF16, device=dev)
        return s
    if op == "ag":
        dt = FP8 if case["dtype"] == "fp8" else BF16
        m, N, K = case["m"], case["N"], case["K"]
        shards = randn(W, m, K, dtype=dt)
        b = randn(N, K, std=0.25 if dt == FP8 else 0.02, dtype=dt).T
        if case["gather"]:      # every rank's shard is an allocation of its own, the gathered matrix and flags are kept
            return dict(s, shards=[shards[r].clone() for r in range(W)], b=b,
                        a_out=torch.empty(W * m, K, dtype=dt, device=dev),
                        progress=torch.zeros(W, dtype=torch.int32, device=dev))
        return dict(s, shards=shards, b=b, a_out=None, progress=None)
    dt = F32 if case["dtype"] == "fp32" else BF16
    M, N, K = case["M"], case["N"], case["K"]
    s["a"] = randn(M, K, dtype=dt)
    s["b"] = randn(N, K, std=0.02, dtype=dt).T if case["b_t"] else randn(K, N, std=0.02, dtype=dt)
    band = M if op == "ar" else M // W
    s["peers"] = randn(W - 1, band, N)
    if op == "ar":
        s["bias"] = randn(N, std=0.02) if case["bias"] else None
    elif op == "rs":
        s["c"] = torch.zeros(M, N, dtype=BF16, device=dev)
    else:
        s["sent"] = torch.zeros(W, band, N, dtype=BF16, device=dev)
    return s


RANK, STRIPE = 1, 2048     # the rank whose work is measured (any W has it), the stripe of interleaved ownership


def _striped_numel(n, W, rank, block):
    full, rest = divmod(n, block * W)
    return full * block + min(block, max(0, rest - rank * block))


# ---- one pass -----------------------------------------------------------------------------------
def run(s):
    op, c = s["op"], s["case"]
    if op == "rms":
        fused.one_shot_all_reduce_bias_rms_norm(s["stack"], s["x"], s["bias"], s["w"], s["y"], rank=RANK)
        return s["y"]
    if op == "norm":
        return fused.rms_norm(s["x"], s["w"])
    if op == "reduce":
        if c["share"] == "all":
            if s["bias"] is None:
                return comm.one_shot_all_reduce(s["stack"])
            fused.one_shot_all_reduce_bias(s["stack"], None, s["bias"], s["out"].view(c["rows"], c["D"]))
            return s["out"]
        if s["bias"] is None:
            return comm.two_shot_all_reduce(s["stack"], rank=RANK, layout=c["share"], BLOCK_SIZE=STRIPE)
        return fused.two_shot_all_reduce_bias(s["stack"], None, s["bias"], s["out"], BLOCK_SIZE=STRIPE, rank=RANK,
                                              layout=c["share"], numel=c["rows"] * c["D"])
    if op == "ag":
        return fused.all_gather_matmul(s["shards"], s["b"], a_out=s["a_out"], progress=s["progress"], rank=RANK,
                                       gather=c["gather"])
    if op == "ar":
        return fused.gemm_one_shot_all_reduce_fused(s["a"], s["b"], peers=s["peers"], bias=s["bias"],
                                                    out_dtype=F32 if c["out"] == "fp32" else BF16)
    if op == "rs":
        return fused.gemm_reduce_scatter(s["a"], s["b"], peers=s["peers"], rank=RANK, c_scratch=s["c"]), s["c"]
    out = fused.gemm_reduce_scatter_ce_persistent(s["a"], s["b"], peers=s["peers"], rank=RANK, sent=s["sent"])
    return out, s["sent"]


# ---- what a pass cannot do without --------------------------------------------------------------
def work(case):
    op, W = case["op"], case["W"]
    if op in ("rms", "norm", "reduce"):
        rows, D = case["rows"], case["D"]
        n = rows * D
        if op == "norm":
            return {"bytes": 2 * (2 * n + D), "flops": 4 * n}
        bias = {"none": 0, "vector": D, "full": n}[case["bias"]]
        if op == "rms":
            return {"bytes": 2 * ((W + 1) * n + bias + D), "flops": (W + 4) * n}
        share = {"all": n, "rows": n // W, "striped": _striped_numel(n, W, RANK, STRIPE)}[case["share"]]
        bias = share if case["bias"] == "full" else bias
        return {"bytes": 2 * ((W + 1) * share + bias), "flops": W * share}
    if op == "ag":
        e = 1 if case["dtype"] == "fp8" else 2
        M, N, K = W * case["m"], case["N"], case["K"]
        copied = M * K if case["gather"] else 0      # the gathered matrix is a result of its own
        return {"bytes": e * (M * K + K * N + M * N + copied), "flops": 2 * M * N * K}
    M, N, K = case["M"], case["N"], case["K"]
    e = 4 if case["dtype"] == "fp32" else 2
    band = M if op == "ar" else M // W
    out = M * N * (4 if op == "ar" and case["out"] == "fp32" else 2)
    return {"bytes": e * (M * K + K * N) + 2 * (W - 1) * band * N + out, "flops": 2 * M * N * K + (W - 1) * band * N}


# ---- how far correct results may be apart -------------------------------------------------------
def tolerance(case):
    op = case["op"]
    if op == "reduce":
        return "exact"            # fp32 sums in a documented order, one rounding
    if op in ("rms", "norm"):
        return {"rel": TOL_ROWS}
    if op == "ag" and case["dtype"] == "fp8":
        return {"rel": TOL_FP8, "max": 0.13}      # a sum next to a rounding boundary goes to the other neighbour, 1/8 away
    if op == "ar" and case["out"] == "fp32":
        return {"rel": TOL_SPLIT if case["dtype"] == "fp32" else TOL_F32}
    return {"rel": TOL_RS_CE if op == "rs_ce" else TOL_BF16}


# Relative errors (2-norm), each about four times what this path showed against the same inputs in 64 bits:
TOL_ROWS = 6.6e-3      # one rounding to bf16: 1.66e-3
TOL_BF16 = 7.6e-3      # one rounding, or two where a product is rounded before the partial sums are added: 1.66e-3 - 1.91e-3
TOL_RS_CE = 1.3e-2     # the copy-engine form adds in bf16, rounding after every rank: 3.3e-3
TOL_F32 = 1.6e-6       # fp32 sums of up to 16384 bf16 products: 4.5e-8 - 4.0e-7
TOL_SPLIT = 1.6e-5     # fp32 operands, 16 mantissa bits of each: 1.5e-6 - 3.8e-6
TOL_FP8 = 3.2e-3       # against the 64-bit sums rounded to fp8: 7.5e-4 - 8.0e-4, 5e-4 of the values one fp8 step off
