"""Operands whose rows start anywhere, laid out anew for the tiled kernel, and outputs whose rows do: every tile, both layouts of B,
every operator and epilogue, gathered operands with odd shares of K and of the rows, one operand in order and the other not.

Operands are small integers, so products and sums over K are exact in fp32 and the outputs are compared bit for bit with the
CPU oracle.  They are views into larger buffers that hold NaN around them: nothing beyond an operand may reach the result.
"""

import pytest
import torch

import iris_amd as iris
from iris_amd import _lib, ops
from helpers import assert_bits_equal, oracle, randint_cpu, randn_cpu, slot_copies, stage_peers

pytestmark = pytest.mark.gpu

FP8 = torch.float8_e4m3fn
# Tile the host picks on 256 CUs -> output size and K: remainders of tiles, of 16-byte pieces and of K steps.
TILES = {"256x256": (4003, 2877, 1003), "128x128_small": (1001, 2877, 2501), "128x128_small2": (1999, 2877, 4003), "64x64": (501, 1501, 5001)}


def _ints(shape, seed, dtype):
    return randint_cpu(shape, seed, torch.float32, -2, 3).to(dtype)


def _view(ctx, value, transposed=False, pad=3):
    v = value.t() if transposed else value
    rows, cols = v.shape
    wide = ctx.zeros((rows + 3, cols + pad), dtype=v.dtype)
    wide.copy_(torch.full((rows + 3, cols + pad), float("nan")).to(v.dtype))
    wide[:rows, :cols].copy_(v)
    view = wide[:rows, :cols]
    return view.t() if transposed else view


def _check(kernel, tile):
    assert kernel.startswith("mfma_") and kernel.endswith("_rows") and tile.split("_")[0] in kernel, kernel


@pytest.mark.parametrize("b_transposed", [False, True], ids=["nn", "nt"])
@pytest.mark.parametrize("tile", sorted(TILES))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, FP8], ids=["bf16", "f16", "fp8"])
def test_every_tile_and_type(dtype, tile, b_transposed):
    M, N, K = TILES[tile]
    out_dtype = torch.bfloat16 if dtype == FP8 else dtype
    ctx = iris.iris(1 << 27, num_ranks=1, rank=0)
    A, B = _ints((M, K), 1, dtype), _ints((K, N), 2, dtype)
    bias = randint_cpu((M,), 3, out_dtype, -8, 9)
    dA, dB, out = _view(ctx, A), _view(ctx, B, b_transposed), ctx.zeros((M, N), dtype=out_dtype)
    for _ in range(2):
        out.fill_(7)
        ops.all_gather_matmul(ctx, out, dA, dB, bias=bias.cuda(), config=iris.FusedConfig(block_size_m=64, block_size_n=64, block_size_k=1))
        _check(_lib.last_kernel(), tile)
        assert_bits_equal(out.cpu(), oracle.all_gather_matmul([A], B, bias=bias, out_dtype=out_dtype), _lib.last_kernel())


@pytest.mark.parametrize("tile,bm,bn", [("64x64", 64, 24), ("64x64", 7, 5), ("128x128_small", 128, 64), ("256x256", 128, 64)])
@pytest.mark.parametrize("op", ["one_shot", "two_shot", "atomic", "reduce_scatter"])
def test_epilogues(op, tile, bm, bn):
    """Flag tiles that pieces straddle (24 and 5 columns), that end inside a piece, and whole ones."""
    W, rank, dtype = (4, 2, torch.bfloat16) if tile == "64x64" else (8, 5, torch.float16)
    M, N, K = TILES[tile]
    ctx = iris.iris(1 << 28, num_ranks=W, rank=rank)
    A, B = _ints((M, K), 5, dtype), _ints((K, N), 6, dtype)
    peers = [randn_cpu((M, N), 40 + r, dtype) for r in range(W)]
    cfg = iris.FusedConfig(block_size_m=bm, block_size_n=bn, block_size_k=1, all_reduce_variant="two_shot" if op == "reduce_scatter" else op)
    dA, dB, dC = _view(ctx, A), _view(ctx, B), ctx.zeros((M, N), dtype=dtype)
    pre, call = (ops.matmul_reduce_scatter_preamble, ops.matmul_reduce_scatter) if op == "reduce_scatter" else (
        ops.matmul_all_reduce_preamble, ops.matmul_all_reduce)
    ws = pre(ctx, dC, dA, dB, config=cfg)
    if op != "atomic":
        stage_peers(ctx, ws, peers)
    for r in range(W):
        ctx.peer_view(dC, r).zero_()
    ws = call(ctx, dC, dA, dB, config=cfg, workspace=ws)
    _check(_lib.last_kernel(), tile)
    got = slot_copies(ctx, dC)
    if op == "atomic":
        for r in range(W):
            assert_bits_equal(got[r] + 0, oracle.gemm(A, B) + 0, f"slot {r}")
        return
    exp = (oracle.matmul_reduce_scatter(A, B, peers, rank, W, bm, bn) if op == "reduce_scatter" else
           oracle.matmul_all_reduce(A, B, peers, rank, W, bm, bn, op))
    assert_bits_equal(ws.aux_buffer.cpu(), exp["aux"], "aux")
    assert torch.equal(ws.locks.cpu(), torch.from_numpy(exp["locks"]))
    for r in range(W) if op == "two_shot" else [rank]:
        assert_bits_equal(got[r], exp["C"][r], f"slot {r}")


@pytest.mark.parametrize("gather_dim,W,M,Kl,N,b_transposed", [
    (1, 3, 501, 1667, 1501, False), (1, 3, 501, 1667, 1501, True), (0, 3, 167, 5001, 1501, False), (0, 2, 256, 5008, 1501, False), (1, 2, 501, 2504, 1501, True)])
def test_gathered_operands(gather_dim, W, M, Kl, N, b_transposed):
    """Odd shares of K per slot (both operands are padded source by source), rows per slot that are no whole tiles; then
    A in order, fetched from the slots as it lies, with only B laid out anew."""
    rank, dtype = W - 1, torch.bfloat16
    ctx = iris.iris(1 << 27, num_ranks=W, rank=rank)
    shards = [_ints((M, Kl), 60 + r, dtype) for r in range(W)]
    K, rows = (W * Kl, M) if gather_dim == 1 else (Kl, W * M)
    B = _ints((K, N), 70, dtype)
    dA = ctx.zeros((M, Kl), dtype=dtype)
    for r in range(W):
        ctx.peer_view(dA, r).copy_(shards[r])
    dB, out = _view(ctx, B, b_transposed), ctx.zeros((rows, N), dtype=dtype)
    ops.all_gather_matmul(ctx, out, dA, dB, config=iris.FusedConfig(block_size_m=1, block_size_n=16, block_size_k=1), gather_dim=gather_dim)
    _check(_lib.last_kernel(), "64x64")
    assert_bits_equal(out.cpu(), oracle.all_gather_matmul(shards, B, gather_dim=gather_dim), _lib.last_kernel())


def test_pushed_rows_streams_and_capture():
    """matmul_all_gather into odd rows of every slot; calls on two streams in turn, each with operands of its own; a captured call
    takes no memory and goes to the any-shape kernel, with the same integers."""
    W, rank, dtype = 2, 1, torch.float16
    M, N, K = TILES["64x64"]
    ctx = iris.iris(1 << 28, num_ranks=W, rank=rank)
    cfg = iris.FusedConfig(block_size_m=1, block_size_n=16, block_size_k=1)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    sets = []
    for i in range(4):
        A, B = _ints((M, K), 80 + 2 * i, dtype), _ints((K, N), 81 + 2 * i, dtype)
        sets.append((_view(ctx, A), _view(ctx, B), ctx.zeros((W * M, N), dtype=dtype), oracle.gemm(A, B)))
    torch.cuda.synchronize()
    for i, (dA, dB, out, _) in enumerate(sets):
        with torch.cuda.stream(streams[i % 2]):
            ops.matmul_all_gather(ctx, out, dA, dB, config=cfg, async_op=True)
            _check(_lib.last_kernel(), "64x64")
    torch.cuda.synchronize()
    for _, _, out, exp in sets:
        for got in slot_copies(ctx, out):
            assert_bits_equal(got[rank * M:(rank + 1) * M], exp, "pushed rows")
    dA, dB, out, exp = sets[0]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.matmul_all_gather(ctx, out, dA, dB, config=cfg, async_op=True)
    assert _lib.last_kernel().startswith("generic_")
    for _ in range(2):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert_bits_equal(out.cpu()[rank * M:(rank + 1) * M], exp, "replayed")
