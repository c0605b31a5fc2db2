"""The end of tiles whose rows start anywhere: last tiles with fewer columns than a 16-byte piece, flag tiles that end inside a
piece of rows that are aligned, numbers of ranks with and without a loop of their own, strided columns.  Operands are small integers
and the outputs are compared bit for bit with the CPU oracle."""

import pytest
import torch

import iris_amd as iris
from iris_amd import _lib, ops
from helpers import assert_bits_equal, heap_tensor, oracle, randint_cpu, randn_cpu, slot_copies, stage_peers

pytestmark = pytest.mark.gpu


def _run(dtype, op, W, M, N, K, bm, bn, strided=False):
    rank = W // 2
    es = 4 if dtype == torch.float32 else 2
    ctx = iris.iris(3 * M * N * es + (M + N) * K * es + (8 << 20), num_ranks=W, rank=rank)
    A, B = randint_cpu((M, K), 1, torch.float32, -2, 3).to(dtype), randint_cpu((K, N), 2, torch.float32, -2, 3).to(dtype)
    peers = [randn_cpu((M, N), 20 + r, dtype) for r in range(W)]
    dA, dB = heap_tensor(ctx, A), heap_tensor(ctx, B)
    memory = ctx.zeros((N, M) if strided else (M, N), dtype=dtype)
    dC = memory.t() if strided else memory
    cfg = iris.FusedConfig(block_size_m=bm, block_size_n=bn, block_size_k=1, all_reduce_variant="two_shot" if op in ("reduce_scatter", "push") else op)
    if op == "push":
        out = ctx.zeros((W * M, N), dtype=dtype)
        ops.matmul_all_gather(ctx, out, dA, dB, config=cfg)
        name = _lib.last_kernel()
        for got in slot_copies(ctx, out):
            assert_bits_equal(got[rank * M:(rank + 1) * M], oracle.gemm(A, B), name)
        return name
    pre, call = (ops.matmul_reduce_scatter_preamble, ops.matmul_reduce_scatter) if op == "reduce_scatter" else (
        ops.matmul_all_reduce_preamble, ops.matmul_all_reduce)
    ws = pre(ctx, dC, dA, dB, config=cfg)
    if op != "atomic":
        # (what a rank publishes lies as C does)
        stage_peers(ctx, ws, [x.t().contiguous().view(M, N) for x in peers] if strided else peers)
    for r in range(W):
        ctx.peer_view(memory, r).zero_()
    ws = call(ctx, dC, dA, dB, config=cfg, workspace=ws)
    name = _lib.last_kernel()
    got = [c.t().contiguous() if strided else c for c in slot_copies(ctx, memory)]
    if op == "atomic":
        for r in range(W):
            assert_bits_equal(got[r] + 0, oracle.gemm(A, B) + 0, f"{name}, slot {r}")
        return name
    exp = (oracle.matmul_reduce_scatter(A, B, peers, rank, W, bm, bn) if op == "reduce_scatter" else
           oracle.matmul_all_reduce(A, B, peers, rank, W, bm, bn, op))
    for again in (False, True):
        if again:  # a workspace handed back: the launch itself leaves zeros in the tiles of others
            memory.fill_(7)
            ws.aux_buffer.fill_(7)
            ws = call(ctx, dC, dA, dB, config=cfg, workspace=ws)
            assert _lib.last_kernel() == name
            got = [c.t().contiguous() if strided else c for c in slot_copies(ctx, memory)]
        aux = ws.aux_buffer.cpu()
        assert_bits_equal(aux.view(N, M).t().contiguous() if strided else aux, exp["aux"], f"{name}, aux")
        assert torch.equal(ws.locks.cpu(), torch.from_numpy(exp["locks"]))
        for r in range(W) if op == "two_shot" else [rank]:
            assert_bits_equal(got[r], exp["C"][r], f"{name}, slot {r}")
    return name


# The last tile has 1 to 7 columns: every tile of the any-shape kernel, and of the tiled one on packed operands.
NARROW = [
    ("generic_bf16_32x32", torch.bfloat16, 60, 67, 24), ("generic_bf16_64x64", torch.bfloat16, 701, 1541, 40),
    ("generic_f16_64x128", torch.float16, 1999, 2819, 24), ("generic_f16_128x128", torch.float16, 2500, 2817, 40),
    ("generic_bf16_256x256", torch.bfloat16, 3900, 3845, 24), ("generic_f32_64x128", torch.float32, 1999, 2819, 12),
    ("mfma_bf16_64x64", torch.bfloat16, 501, 1541, 5001), ("mfma_f16_128x128", torch.float16, 1001, 2819, 2501), ("mfma_bf16_256x256", torch.bfloat16, 4003, 2821, 1003),
]


@pytest.mark.parametrize("op,W", [("one_shot", 8), ("one_shot", 3), ("two_shot", 4), ("reduce_scatter", 2), ("two_shot", 9), ("atomic", 2), ("push", 2)])
@pytest.mark.parametrize("kernel,dtype,M,N,K", NARROW, ids=[c[0] for c in NARROW])
def test_last_tiles_narrower_than_a_piece(kernel, dtype, M, N, K, op, W):
    if W > 4 and M > 2000:
        W = 4
    name = _run(dtype, op, W, M, N, K, 32, 64)
    assert name.startswith(kernel) or W in (3, 9), name


# Two columns behind the last edge of a flag tile: the last piece of a row is moved to the left over that edge.
@pytest.mark.parametrize("op,W", [("two_shot", 4), ("reduce_scatter", 2), ("two_shot", 3)])
@pytest.mark.parametrize("kernel,dtype,M,K", [("generic_bf16_64x128", torch.bfloat16, 1999, 24), ("generic_f32_64x128", torch.float32, 1999, 12),
                                              ("mfma_f16_128x128", torch.float16, 1001, 2501), ("mfma_bf16_256x256", torch.bfloat16, 4003, 1003)])
def test_last_piece_over_the_edge_of_a_flag_tile(kernel, dtype, M, K, op, W):
    name = _run(dtype, op, W, M, 2882, K, 32, 64)
    assert name.startswith(kernel) or W == 3, name


@pytest.mark.parametrize("op", ["two_shot", "reduce_scatter"])
@pytest.mark.parametrize("dtype,N,bn", [(torch.bfloat16, 2824, 100), (torch.float32, 2820, 70), (torch.float16, 2816, 12), (torch.bfloat16, 2824, 104),
                                        (torch.bfloat16, 2877, 100), (torch.float32, 2877, 70), (torch.float16, 2877, 12), (torch.bfloat16, 1501, 5)])
def test_flag_tiles_that_end_inside_a_piece(op, dtype, N, bn):
    _run(dtype, op, 8, 1000, N, 24, 64, bn)


# Both ways to read the peers' tiles, from other numbers of ranks than 2, 4 and 8 (the line lies at 32 MiB read).
@pytest.mark.parametrize("W,M,N", [(3, 1000, 2877), (3, 4000, 2877), (6, 2000, 2877), (6, 1000, 2875), (9, 900, 2877)])
def test_any_number_of_ranks_on_both_sides_of_the_line(W, M, N):
    _run(torch.bfloat16, "one_shot", W, M, N, 17, 128, 64)
    _run(torch.bfloat16, "one_shot", W, M, N // 16 * 16, 32, 128, 64)  # tiled kernel


@pytest.mark.parametrize("op", ["one_shot", "two_shot", "reduce_scatter", "atomic"])
def test_strided_columns(op):
    _run(torch.bfloat16, op, 4, 301, 517, 40, 64, 24, strided=True)
