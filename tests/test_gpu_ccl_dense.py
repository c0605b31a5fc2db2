"""One-shot all-reduce of dense tensors (dense_sum_kernel of iris_ccl.hip): ranks added in ascending order in float32
from +0 and rounded once, so every comparison is bit for bit."""

import pytest
import torch

import iris_amd as iris
from iris_amd import _lib
from iris_amd.ccl import Config
from helpers import assert_bits_equal, randn_cpu

pytestmark = pytest.mark.gpu


# One chunk; the last thread of a workgroup and the first of the next; more chunks than one pass of the grid has threads
# (two ranks, below the size that streams); streamed, with a last group of four that is not full, and several passes.
@pytest.mark.parametrize("W,rank,M,N,dtype", [
    (2, 1, 1, 8, torch.bfloat16), (4, 0, 1, 4, torch.float32), (8, 5, 1, 128 * 8, torch.float16), (8, 7, 1, 129 * 8, torch.bfloat16),
    (4, 3, 127, 1016, torch.float16), (2, 0, 1100, 4096, torch.bfloat16), (8, 2, 1025, 2888, torch.bfloat16),
    (4, 1, 1999, 2052, torch.float32), (2, 1, 3000, 8192, torch.float16)])
def test_dense_one_shot(W, rank, M, N, dtype):
    es = torch.empty((), dtype=dtype).element_size()
    ctx = iris.iris(2 * M * N * es + (1 << 21), num_ranks=W, rank=rank)
    x, y = ctx.zeros((M, N), dtype=dtype), ctx.zeros((M, N), dtype=dtype)
    inputs = [randn_cpu((M, N), 7 + r, dtype) for r in range(W)]
    inputs[0][0, 0] = -0.0  # +0 + -0 is +0
    for r in range(1, W):
        inputs[r][0, 0] = -0.0
    inputs[W - 1][-1, -1] = float("inf")
    for r in range(W):
        ctx.peer_view(x, r).copy_(inputs[r])
        ctx.peer_view(y, r).fill_(3.0)
    ctx.ccl.all_reduce(y, x, config=Config(all_reduce_variant="one_shot"))
    assert _lib.last_kernel().startswith("dense_sum_one_shot_"), _lib.last_kernel()
    exp = torch.zeros((M, N))
    for r in range(W):
        exp += inputs[r].float()
    assert_bits_equal(y.cpu(), exp.to(dtype), f"{W} ranks, {M}x{N}")
    for r in range(W):
        assert_bits_equal(ctx.peer_view(x, r).cpu(), inputs[r], f"input of slot {r}")
        if r != rank:
            assert bool((ctx.peer_view(y, r) == 3.0).all()), f"output of slot {r} was written"


def _staged(W, rank, M, N, dtype, row=None):
    """Inputs of all ranks in one heap, rows `row` elements apart; outputs filled with 3."""
    row = row or N
    ctx = iris.iris(1 << 24, num_ranks=W, rank=rank)
    x, y = ctx.zeros((M, row), dtype=dtype), ctx.zeros((M, row), dtype=dtype)
    inputs = [randn_cpu((M, N), 70 + r, dtype) for r in range(W)]
    for r in range(W):
        ctx.peer_view(x, r)[:, :N].copy_(inputs[r])
        ctx.peer_view(y, r).fill_(3.0)
    return ctx, x, y, inputs


def _sum(inputs, dtype):
    exp = torch.zeros(inputs[0].shape)
    for t in inputs:
        exp += t.float()
    return exp.to(dtype)


# Members between outsiders; two members that start past rank 0; four next to each other.
@pytest.mark.parametrize("W,rank,group,dtype", [
    (8, 5, [1, 3, 5, 7], torch.bfloat16), (8, 6, [2, 6], torch.float32), (8, 2, [2, 3, 4, 5], torch.float16)])
def test_dense_one_shot_of_a_group(W, rank, group, dtype):
    ctx, x, y, inputs = _staged(W, rank, 33, 264, dtype)
    outsiders = [r for r in range(W) if r not in group]
    for r in outsiders:
        ctx.peer_view(x, r).fill_(float("nan"))
    ctx.ccl.all_reduce(y, x, group=group, config=Config(all_reduce_variant="one_shot"))
    assert _lib.last_kernel().startswith("dense_sum_one_shot_"), _lib.last_kernel()
    assert_bits_equal(y.cpu(), _sum([inputs[r] for r in group], dtype), f"group {group}")
    for r in range(W):
        if r != rank:
            assert bool((ctx.peer_view(y, r) == 3.0).all()), f"output of slot {r} was written"


@pytest.mark.parametrize("M,N", [(5, 136), (2048, 4096)])  # the second one streams, four chunks to a thread
def test_dense_one_shot_in_place(M, N):
    W, rank, dtype = 8, 3, torch.bfloat16
    ctx = iris.iris(2 * M * N * 2 + (1 << 21), num_ranks=W, rank=rank)
    x, other = ctx.zeros((M, N), dtype=dtype), ctx.zeros((M, N), dtype=dtype)
    inputs = [randn_cpu((M, N), 90 + r, dtype) for r in range(W)]
    for r in range(W):
        ctx.peer_view(x, r).copy_(inputs[r])
    cfg = Config(all_reduce_variant="one_shot")
    ws = ctx.ccl.all_reduce_preamble(other, x, config=cfg)  # (it zeroes the output it is given)
    ctx.ccl.all_reduce(x, x, config=cfg, workspace=ws)
    assert _lib.last_kernel().startswith("dense_sum_one_shot_"), _lib.last_kernel()
    assert_bits_equal(x.cpu(), _sum(inputs, dtype), "in place")


# What the dense kernel does not take: a group size it is not built for, rows with space between them, and rows that are not
# whole chunks.
@pytest.mark.parametrize("W,rank,N,row", [(3, 1, 256, 256), (1, 0, 256, 256), (4, 2, 256, 264), (4, 2, 250, 250)])
def test_other_one_shots_run_the_general_kernel(W, rank, N, row):
    dtype = torch.float16
    ctx, x, y, inputs = _staged(W, rank, 21, N, dtype, row)
    y = y[:, :N]
    ctx.ccl.all_reduce(y, x[:, :N], config=Config(all_reduce_variant="one_shot"))
    assert _lib.last_kernel().startswith("slot_reduce_one_shot_"), _lib.last_kernel()
    assert_bits_equal(y.cpu(), _sum(inputs, dtype), f"{W} ranks, {N} columns, rows {row} apart")


# Eight ranks and 16-bit data on both sides of 512 MiB of traffic (nine tensors); float32 stays with the dense kernel.
@pytest.mark.parametrize("M,dtype,kernel", [
    (7281, torch.bfloat16, "dense_sum"), (7282, torch.bfloat16, "slot_reduce"), (7282, torch.float16, "slot_reduce"),
    (3641, torch.float32, "dense_sum")])
def test_large_dense_one_shots_of_eight_ranks(M, dtype, kernel):
    W, rank, N = 8, 6, 4096
    es = torch.empty((), dtype=dtype).element_size()
    ctx = iris.iris(2 * M * N * es + (1 << 21), num_ranks=W, rank=rank)
    x, y = ctx.zeros((M, N), dtype=dtype), ctx.zeros((M, N), dtype=dtype)
    exp = torch.zeros((M, N), device="cuda")
    for r in range(W):
        g = torch.Generator(device="cuda").manual_seed(50 + r)
        data = torch.randn((M, N), generator=g, device="cuda").to(dtype)
        ctx.peer_view(x, r).copy_(data)
        exp += data.float()
    ctx.ccl.all_reduce(y, x, config=Config(all_reduce_variant="one_shot"))
    assert _lib.last_kernel().startswith(kernel), _lib.last_kernel()
    assert torch.equal(y, exp.to(dtype))
