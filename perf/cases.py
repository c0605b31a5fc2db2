"""Calls that programs on this framework make, with inputs of the sizes they make them with.

One process plays one rank of a W-rank tensor-parallel job (the other ranks' heap slots are staged once, as
the peers would have left them) and calls the operators as its layers come by: the workspace of the
layer is kept and handed back in, the host does not wait between calls.  Sizes are those of the
repository's benchmark grids (N = 2880 and 3584, K = 4096 / W, 1376, 8192), of bench.py and of the tests; drawn cases
spread over the ranges between them.

    listed()          the named cases
    draw(rng)         one more case of the same ranges
    prepare(case, s)  context, inputs of seed s, workspace
    run(state)        one call of the operator; returns every buffer that the call writes
    work(case)        compulsory bytes and flops of one call
    tolerance(case)   how far another correct implementation may be off
"""

import math

import torch

import iris_amd as iris
from iris_amd.ccl import Config
from iris_amd.ops import matmul_all_reduce_preamble, matmul_reduce_scatter_preamble

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32, "fp8": torch.float8_e4m3fn}
_BYTES = {"bf16": 2, "fp16": 2, "fp32": 4, "fp8": 1}


def _out(case):
    return "bf16" if case["dtype"] == "fp8" else case["dtype"]


def listed():
    return [
        # A decode step: 32 tokens through a row-parallel projection, latency decides.
        dict(name="decode_one_shot_fp16", op="matmul_all_reduce", variant="one_shot", dtype="fp16", W=8, rank=0, M=32, N=2880, K=512, bm=32),
        # The same layer when prompts and decodes share a batch; the default variant of the operator.
        dict(name="hybrid_two_shot_fp16", op="matmul_all_reduce", variant="two_shot", dtype="fp16", W=8, rank=0, M=896, N=2880, K=512, bm=128),
        # The default workload of bench.py: prefill of 4096 tokens.
        dict(name="prefill_one_shot_bf16", op="matmul_all_reduce", variant="one_shot", dtype="bf16", W=8, rank=0, M=4096, N=4096, K=1376, bm=256),
        # The largest call: 16384 tokens, e4m3 operands with per-tensor scales.
        dict(name="prefill_one_shot_fp8", op="matmul_all_reduce", variant="one_shot", dtype="fp8", W=8, rank=0, M=16384, N=8192, K=1024, bm=256),
        # float32 data, as in numerics checks and in layers kept at full precision.
        dict(name="float32_two_shot", op="matmul_all_reduce", variant="two_shot", dtype="fp32", W=4, rank=1, M=2048, N=2880, K=1024, bm=128),
        # Nothing is a multiple of anything: a vocabulary-like N and an unpadded K.
        dict(name="ragged_one_shot_bf16", op="matmul_all_reduce", variant="one_shot", dtype="bf16", W=8, rank=0, M=1999, N=2877, K=1371, bm=128),
        # Sequence-parallel input, gathered by rows into a column-parallel projection.
        dict(name="row_gather_bf16", op="all_gather_matmul", gather=0, bias=False, dtype="bf16", W=8, rank=0, M=8192, N=1792, K=4096, bm=256),
        # The reference's layout: columns of A on the ranks, with the row bias.
        dict(name="column_gather_fp16", op="all_gather_matmul", gather=1, bias=True, dtype="fp16", W=8, rank=0, M=4096, N=3584, K=8192, bm=256),
        # The product of this rank's rows, pushed to everybody.
        dict(name="push_gather_fp16", op="matmul_all_gather", bias=False, dtype="fp16", W=4, rank=1, M=1024, N=3584, K=8192, bm=256),
        # Row-parallel projection back into sequence shards.
        dict(name="reduce_scatter_bf16", op="matmul_reduce_scatter", dtype="bf16", W=8, rank=0, M=8192, N=4096, K=1376, bm=256),
        # The stand-alone all-reduce behind a library GEMM, a prefill and a decode step.
        dict(name="ccl_two_shot_bf16", op="ccl_all_reduce", variant="two_shot", dtype="bf16", W=8, rank=0, M=8192, N=2880),
        dict(name="ccl_one_shot_decode_bf16", op="ccl_all_reduce", variant="one_shot", dtype="bf16", W=8, rank=0, M=64, N=2880),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["matmul_all_reduce", "matmul_all_reduce", "all_gather_matmul", "matmul_all_gather", "matmul_reduce_scatter",
                     "ccl_all_reduce", "ccl_reduce_scatter"])
    W = rng.choice([2, 4, 8, 8])
    case = dict(op=op, W=W, rank=rng.randrange(W))
    ragged = rng.random() < 0.3  # N and K as they come, instead of whole 16-byte pieces
    if op.startswith("ccl_"):
        case["dtype"] = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        case["M"], case["N"] = _log_uniform(rng, 1, 16384), _log_uniform(rng, 64, 8192)
        if op == "ccl_all_reduce":
            case["variant"] = rng.choice(["one_shot", "two_shot"])
        if not ragged:
            case["N"] = max(case["N"] // 16, 4) * 16
        return case
    case["dtype"] = rng.choice(["bf16", "bf16", "fp16", "fp16", "fp8", "fp32"])
    if op == "matmul_all_reduce":
        case["variant"] = rng.choice(["one_shot", "two_shot", "two_shot", "atomic"])
    if op == "all_gather_matmul":
        case["gather"] = rng.choice([0, 1])
    if op in ("all_gather_matmul", "matmul_all_gather"):
        case["bias"] = rng.random() < 0.5
    while True:
        M, N, K = _log_uniform(rng, 1, 16384), _log_uniform(rng, 64, 8192), _log_uniform(rng, 64, 8192)
        if not ragged:
            N, K = max(N // 16, 4) * 16, max(K // 16, 4) * 16
        if case.get("gather") == 0:
            M = max(M // W, 1) * W
        if case.get("gather") == 1:  # every rank holds K / W columns
            K = max(K // W, 32) * W if ragged else max(K // W // 16, 4) * 16 * W
        # No dearer than the largest listed case; float32 and ragged cases a quarter of its flops.
        if 2 * M * N * K <= (6e10 if ragged or case["dtype"] == "fp32" else 2.7e11) and W * M * N <= 2.7e8:
            break
    case["M"], case["N"], case["K"] = M, N, K
    rows = M // W if case.get("gather") == 0 else M
    case["bm"] = next(b for b in (256, 128, 64, 32, 16, 8, 4, 2, 1) if b <= rows)
    return case


def _randn(shape, gen, dtype, scale=1.0):
    """N(0, scale) in `dtype`; e4m3 values are returned with the scale that takes them back."""
    x = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32 if dtype == "fp8" else _DTYPES[dtype])
    if dtype != "fp8":
        return x.mul_(scale), None
    amax = float(x.abs().max()) / 448.0
    return x.div_(amax).to(_DTYPES[dtype]), amax


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    W, rank, M, N = case["W"], case["rank"], case["M"], case["N"]
    out = _out(case)
    es = _BYTES[out]
    if case["op"].startswith("ccl_"):
        ctx = iris.iris(2 * M * N * es + (1 << 20), num_ranks=W, rank=rank)
        x, y = ctx.zeros((M, N), dtype=_DTYPES[out]), ctx.zeros((M, N), dtype=_DTYPES[out])
        for r in range(W):
            ctx.peer_view(x, r).copy_(_randn((M, N), gen, out)[0])
        s = dict(case=case, ctx=ctx, x=x, y=y, ws=None)
        s["config"] = Config(all_reduce_variant=case["variant"]) if "variant" in case else Config()
        if case["op"] == "ccl_all_reduce":
            s["ws"] = ctx.ccl.all_reduce_preamble(y, x, config=s["config"])
        s["out"] = [ctx.peer_view(y, r) for r in range(W)] if case.get("variant") == "two_shot" else [y]
        torch.cuda.synchronize()
        return s

    K, dtype = case["K"], case["dtype"]
    a_rows, a_cols = M, K
    if case.get("gather") == 0:
        a_rows = M // W
    if case.get("gather") == 1:
        a_cols = K // W
    c_rows = M * W if case["op"] == "matmul_all_gather" else M
    outputs = 2 if case["op"] in ("matmul_all_reduce", "matmul_reduce_scatter") else 1  # C, and what the rank publishes
    ctx = iris.iris((a_rows * a_cols + K * N) * _BYTES[dtype] + outputs * c_rows * N * es + (4 << 20), num_ranks=W, rank=rank)
    config = iris.FusedConfig(block_size_m=case["bm"], block_size_n=64, block_size_k=32, all_reduce_variant=case.get("variant", "two_shot"))
    A, B = ctx.zeros((a_rows, a_cols), dtype=_DTYPES[dtype]), ctx.zeros((K, N), dtype=_DTYPES[dtype])
    C = ctx.zeros((c_rows, N), dtype=_DTYPES[out])
    a, scale_a = _randn((a_rows, a_cols), gen, dtype, K ** -0.5)
    A.copy_(a)
    for r in range(W if "gather" in case else 0):  # every rank's shard of A, quantised with one scale
        if r != rank:
            x = torch.randn((a_rows, a_cols), generator=gen, device="cuda")
            x = x.div_(scale_a).clamp_(-448.0, 448.0) if scale_a else x.mul_(K ** -0.5)
            ctx.peer_view(A, r).copy_(x)
    b, scale_b = _randn((K, N), gen, dtype)
    B.copy_(b)
    s = dict(case=case, ctx=ctx, config=config, A=A, B=B, C=C, ws=None, bias=None)
    s["scales"] = dict(scale_a=scale_a, scale_b=scale_b) if scale_a else {}
    if case.get("bias"):
        s["bias"] = _randn((M,), gen, out)[0]
    if case["op"] == "matmul_all_reduce":
        s["ws"] = matmul_all_reduce_preamble(ctx, C, A, B, config=config)
    elif case["op"] == "matmul_reduce_scatter":
        s["ws"] = matmul_reduce_scatter_preamble(ctx, C, A, B, config)
    if s["ws"] is not None and s["ws"].aux_buffer is not None:
        for r in range(W):  # the peers have published their products and raised their flags
            if r != rank:
                ctx.peer_view(s["ws"].aux_buffer, r).copy_(_randn((M, N), gen, out)[0])
                ctx.peer_view(s["ws"].locks, r).fill_(1)
    everywhere = case["op"] == "matmul_all_gather" or case.get("variant") == "two_shot"
    s["out"] = [ctx.peer_view(C, r) for r in range(W)] if everywhere else [C]
    if s["ws"] is not None and s["ws"].aux_buffer is not None:
        s["out"] += [s["ws"].aux_buffer, s["ws"].locks]
    torch.cuda.synchronize()
    return s


def run(s):
    ops, op = s["ctx"].ops, s["case"]["op"]
    if op == "matmul_all_reduce":
        s["ws"] = ops.matmul_all_reduce(s["C"], s["A"], s["B"], async_op=True, config=s["config"], workspace=s["ws"], **s["scales"])
    elif op == "matmul_reduce_scatter":
        s["ws"] = ops.matmul_reduce_scatter(s["C"], s["A"], s["B"], async_op=True, config=s["config"], workspace=s["ws"], **s["scales"])
    elif op == "all_gather_matmul":
        ops.all_gather_matmul(s["C"], s["A"], s["B"], bias=s["bias"], async_op=True, config=s["config"], gather_dim=s["case"]["gather"], **s["scales"])
    elif op == "matmul_all_gather":
        ops.matmul_all_gather(s["C"], s["A"], s["B"], bias=s["bias"], async_op=True, config=s["config"], **s["scales"])
    elif op == "ccl_all_reduce":
        s["ws"] = s["ctx"].ccl.all_reduce(s["y"], s["x"], async_op=True, config=s["config"], workspace=s["ws"])
    else:
        s["ctx"].ccl.reduce_scatter(s["y"], s["x"], async_op=True, config=s["config"])
    return s["out"]


def work(case):
    """Operands read once, the peers' partial results that this rank sums read once, results written once."""
    W, mn = case["W"], case["M"] * case["N"]
    es = _BYTES[_out(case)]
    variant = case.get("variant", "")
    share = 1 if variant == "one_shot" else 1 / W  # of the tiles, reduced by this rank
    stores = W if variant == "two_shot" else 1
    if case["op"].startswith("ccl_"):
        return {"bytes": int(mn * es * share * (W + stores)), "flops": int(mn * share * (W - 1))}
    flops = 2 * mn * case["K"]
    a_and_b = (case["M"] * case["K"] + case["K"] * case["N"]) * _BYTES[case["dtype"]]
    if case["op"] == "all_gather_matmul":
        bytes_ = mn * es
    elif case["op"] == "matmul_all_gather":
        bytes_ = W * mn * es
    elif variant == "atomic":
        bytes_ = 2 * W * mn * es
    else:  # own product published, peers' products of the owned tiles read, sums stored
        bytes_ = mn * es + int(mn * es * share * (W - 1 + stores))
    return {"bytes": a_and_b + bytes_, "flops": flops}


# (relative 2-norm, largest difference) by type of the operands.  Measured against products and sums in 64
# bits, rounded where the kernels round: bf16 4e-5 and 0.008 (a sum that falls on the other side of a rounding
# boundary moves one value by 2^-8; the matrix of a product and the sums of it both round), fp16 1.7e-5
# and 0.001, e4m3 operands 2.3e-4 and 0.016, float32 6e-7 and 5e-6 at K = 1024.  Four times that for the
# largest difference; the 2-norm leaves room for one such value in an output of a few dozen (and
# float32 for sums over eight times the K).
_TOLERANCE = {"bf16": (2e-3, 0.032), "fp16": (2.5e-4, 0.004), "fp8": (2e-3, 0.064), "fp32": (5e-6, 6e-5)}


def tolerance(case):
    if case["op"].startswith("ccl_"):
        return "exact"  # the order of the fp32 additions is part of these collectives' contract
    rel, most = _TOLERANCE[case["dtype"]]
    return {"rel": rel, "max": most}
