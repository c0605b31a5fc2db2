"""Operands laid out anew and the any-shape kernel, which takes the same launches when there is no memory for that, give the same
bits: random data, so that another order of the fp32 sums shows."""

import pytest
import torch

import iris_amd as iris
from iris_amd import _lib, ops
from helpers import heap_tensor, randn_cpu, stage_peers

pytestmark = pytest.mark.gpu

FP8 = torch.float8_e4m3fn
TILES = {"256x256": (4003, 2877, 1003), "128x128": (1001, 2877, 2501), "64x64": (501, 1501, 5001)}


def _same(call, out):
    """Both kernels, in turn, into the same output."""
    got = []
    for path in ("auto", "generic", "auto"):
        out.fill_(3)
        call(path)
        name = _lib.last_kernel()
        assert name.endswith("_rows") if path == "auto" else name.startswith("generic_"), name
        got.append(out.cpu().view(torch.int16))
    assert torch.isfinite(out.float()).all()
    assert torch.equal(got[0], got[2])
    differ = int((got[0] != got[1]).sum())
    assert differ == 0, f"{differ} of {got[0].numel()} values differ"


@pytest.mark.parametrize("b_transposed", [False, True], ids=["nn", "nt"])
@pytest.mark.parametrize("tile", sorted(TILES))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, FP8], ids=["bf16", "f16", "fp8"])
def test_every_tile_and_type(dtype, tile, b_transposed):
    M, N, K = TILES[tile]
    out_dtype = torch.bfloat16 if dtype == FP8 else dtype
    ctx = iris.iris(1 << 27, num_ranks=1, rank=0)
    A, B = randn_cpu((M, K), 1, dtype, K ** -0.5 if dtype != FP8 else 1.0), randn_cpu((N, K) if b_transposed else (K, N), 2, dtype)
    dA, dB, out = heap_tensor(ctx, A), heap_tensor(ctx, B), ctx.zeros((M, N), dtype=out_dtype)
    bias = randn_cpu((M,), 3, out_dtype).cuda()
    scales = dict(scale_a=0.3, scale_b=0.01) if dtype == FP8 else {}
    cfg = iris.FusedConfig(block_size_m=64, block_size_n=64, block_size_k=1)
    _same(lambda path: ops.all_gather_matmul(ctx, out, dA, dB.t() if b_transposed else dB, bias=bias, config=cfg, kernel_path=path, **scales), out)


# Shares of K that end inside a 16-byte piece, and on one but inside a matrix product (2504 = 156 * 16 + 8): laid out, the next
# source follows there.
@pytest.mark.parametrize("W,M,Kl,N,dtype", [(3, 501, 1667, 1501, torch.bfloat16), (2, 501, 2504, 1501, torch.float16), (4, 4003, 251, 2877, torch.bfloat16),
                                            (2, 1001, 1251, 2877, FP8), (8, 1001, 313, 2877, torch.float16)])
@pytest.mark.parametrize("b_transposed", [False, True], ids=["nn", "nt"])
def test_columns_gathered_from_every_rank(W, M, Kl, N, dtype, b_transposed):
    out_dtype = torch.bfloat16 if dtype == FP8 else dtype
    K, rank = W * Kl, W - 1
    ctx = iris.iris(1 << 27, num_ranks=W, rank=rank)
    base = ctx.zeros((M + 1, Kl), dtype=dtype)  # rows start off 16 bytes, also where Kl is whole pieces
    dA = base.view(-1)[1:1 + M * Kl].view(M, Kl)
    for r in range(W):
        ctx.peer_view(base, r).view(-1)[1:1 + M * Kl].view(M, Kl).copy_(randn_cpu((M, Kl), 10 + r, dtype, 1.0 if dtype == FP8 else K ** -0.5))
    B = heap_tensor(ctx, randn_cpu((N, K) if b_transposed else (K, N), 2, dtype))
    out = ctx.zeros((M, N), dtype=out_dtype)
    cfg = iris.FusedConfig(block_size_m=1, block_size_n=16, block_size_k=1)
    _same(lambda path: ops.all_gather_matmul(ctx, out, dA, B.t() if b_transposed else B, config=cfg, gather_dim=1, kernel_path=path), out)


@pytest.mark.parametrize("variant", ["one_shot", "two_shot"])
def test_eager_and_captured_calls_agree(variant):
    """A captured call takes no memory: another kernel, the same bits, in every replay."""
    W, rank, dtype = 4, 1, torch.bfloat16
    M, N, K = TILES["256x256"]
    ctx = iris.iris(1 << 27, num_ranks=W, rank=rank)
    dA, dB, dC = heap_tensor(ctx, randn_cpu((M, K), 1, dtype, K ** -0.5)), heap_tensor(ctx, randn_cpu((K, N), 2, dtype)), ctx.zeros((M, N), dtype=dtype)
    cfg = iris.FusedConfig(block_size_m=128, block_size_n=64, block_size_k=1, all_reduce_variant=variant)
    ws = ops.matmul_all_reduce_preamble(ctx, dC, dA, dB, config=cfg)
    stage_peers(ctx, ws, [randn_cpu((M, N), 20 + r, dtype) for r in range(W)])
    ops.matmul_all_reduce(ctx, dC, dA, dB, config=cfg, workspace=ws, async_op=True)
    assert _lib.last_kernel().endswith("_rows")
    torch.cuda.synchronize()
    want = dC.cpu().view(torch.int16)
    ws = ops.matmul_all_reduce_preamble(ctx, dC, dA, dB, config=cfg)
    stage_peers(ctx, ws, [randn_cpu((M, N), 20 + r, dtype) for r in range(W)])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.matmul_all_reduce(ctx, dC, dA, dB, config=cfg, workspace=ws, async_op=True)
    assert _lib.last_kernel().startswith("generic_")
    dC.zero_()
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(dC.cpu().view(torch.int16), want)


def test_tiles_that_split_k_stay_on_the_any_shape_kernel():
    """32x32 tiles of the any-shape kernel add four partial sums over K, whatever memory there is."""
    cfg = iris.FusedConfig(block_size_m=1, block_size_n=16, block_size_k=1)
    M, N, K = 156, 1797, 4496
    ctx = iris.iris(1 << 27, num_ranks=1, rank=0)
    dA, dB, out = heap_tensor(ctx, randn_cpu((M, K), 1, torch.bfloat16)), heap_tensor(ctx, randn_cpu((N, K), 2, torch.bfloat16)), ctx.zeros((M, N), dtype=torch.bfloat16)
    ops.all_gather_matmul(ctx, out, dA, dB.t(), config=cfg)
    assert _lib.last_kernel() == "generic_bf16_32x32_nt", _lib.last_kernel()
    M, N, K = 70, 4336, 6575
    ctx = iris.iris(1 << 27, num_ranks=2, rank=1)
    dA, dB, out = heap_tensor(ctx, randn_cpu((M, K), 1, torch.float16)), heap_tensor(ctx, randn_cpu((K, N), 2, torch.float16)), ctx.zeros((2 * M, N), dtype=torch.float16)
    ops.matmul_all_gather(ctx, out, dA, dB, config=cfg)
    assert _lib.last_kernel() == "generic_f16_32x32_nn", _lib.last_kernel()


# What packing costs more than it gives: a short K on 128x128 tiles, more 128x128 or 64x64 tiles than CUs, sums of three ranks; and the
# other side of each line.
@pytest.mark.parametrize("op,W,M,N,K,packed", [
    ("plain", 1, 1001, 2877, 2301, False), ("plain", 1, 1001, 2877, 2501, True), ("plain", 1, 1999, 2877, 3501, False),
    ("plain", 1, 1999, 2877, 4003, True), ("plain", 1, 2999, 2877, 4003, True), ("plain", 1, 1501, 2877, 4003, False),
    ("plain", 1, 501, 2301, 5001, False), ("plain", 1, 501, 1501, 5001, True), ("one_shot", 3, 4003, 2877, 1003, False), ("one_shot", 2, 4003, 2877, 1003, True)])
def test_where_operands_are_laid_out_anew(op, W, M, N, K, packed):
    dtype = torch.bfloat16
    ctx = iris.iris(1 << 28, num_ranks=W, rank=W - 1)
    dA, dB, out = ctx.zeros((M, K), dtype=dtype), ctx.zeros((K, N), dtype=dtype), ctx.zeros((M, N), dtype=dtype)
    cfg = iris.FusedConfig(block_size_m=64, block_size_n=64, block_size_k=1, all_reduce_variant="one_shot")
    if op == "plain":
        ops.all_gather_matmul(ctx, out, dA, dB, config=cfg)
    else:
        ws = ops.matmul_all_reduce_preamble(ctx, out, dA, dB, config=cfg)
        stage_peers(ctx, ws, [torch.zeros((M, N), dtype=dtype) for _ in range(W)])
        ops.matmul_all_reduce(ctx, out, dA, dB, config=cfg, workspace=ws)
    assert _lib.last_kernel().endswith("_rows") == packed, _lib.last_kernel()
    assert not out.any()
