"""The end of tiles whose rows start anywhere: flag tiles that end inside a piece of rows that are aligned, numbers of
ranks with and without a loop of their own.  Operands are small integers
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
    aux = ws.aux_buffer.cpu()
    assert_bits_equal(aux.view(N, M).t().contiguous() if strided else aux, exp["aux"], f"{name}, aux")
    assert torch.equal(ws.locks.cpu(), torch.from_numpy(exp["locks"]))
    for r in range(W) if op == "two_shot" else [rank]:
        assert_bits_equal(got[r], exp["C"][r], f"{name}, slot {r}")
    return name


@pytest.mark.parametrize("op", ["two_shot", "reduce_scatter"])
@pytest.mark.parametrize("dtype,N,bn", [(torch.bfloat16, 2824, 100), (torch.float32, 2820, 70), (torch.float16, 2816, 12), (torch.bfloat16, 2824, 104)])
def test_flag_tiles_that_end_inside_a_piece_of_aligned_rows(op, dtype, N, bn):
    _run(dtype, op, 8, 1000, N, 24, 64, bn)


# Both ways to read the peers' tiles, from other numbers of ranks than 2, 4 and 8 (the line lies at 32 MiB read).
@pytest.mark.parametrize("W,M,N", [(3, 1000, 2877), (3, 4000, 2877), (6, 2000, 2877), (6, 1000, 2875), (9, 900, 2877)])
def test_any_number_of_ranks_on_both_sides_of_the_line(W, M, N):
    _run(torch.bfloat16, "one_shot", W, M, N, 17, 128, 64)
    _run(torch.bfloat16, "one_shot", W, M, N // 16 * 16, 32, 128, 64)  # tiled kernel
