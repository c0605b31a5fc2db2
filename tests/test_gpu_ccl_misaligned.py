"""The stand-alone collectives on rows that are not whole 16-byte chunks, against the CPU oracle, bit for bit."""

import pytest
import torch

import iris_amd as iris
from iris_amd import _lib
from iris_amd.ccl import Config
from helpers import assert_bits_equal, oracle, randn_cpu

pytestmark = pytest.mark.gpu


def _stage(ctx, inputs, out_fill=0.0):
    """Heap tensors for input and output with every slot filled."""
    d_in, d_out = (ctx.zeros(tuple(inputs[0].shape), dtype=inputs[0].dtype) for _ in range(2))
    for r, value in enumerate(inputs):
        ctx.peer_view(d_in, r).copy_(value)
        ctx.peer_view(d_out, r).fill_(out_fill)
    return d_in, d_out


@pytest.mark.parametrize("variant", ["one_shot", "reduce_scatter", "two_shot"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N", [(70, 51), (1, 9), (3, 8), (33, 321), (2100, 2881)])
def test_misaligned_rows(dtype, variant, M, N):
    """Rows that start anywhere and a last 16-byte chunk that starts inside its neighbour, on small and on streamed
    sizes; the last tile column of N = 321 has one column."""
    W, rank = 4, 1
    ctx = iris.iris(1 << 26, num_ranks=W, rank=rank)
    inputs = [randn_cpu((M, N), 70 + r, dtype) for r in range(W)]
    d_in, d_out = _stage(ctx, inputs, out_fill=5.0)
    filled = torch.full((M, N), 5.0, dtype=dtype)
    if variant == "reduce_scatter":
        ctx.ccl.reduce_scatter(d_out, d_in, config=Config())
        exp = oracle.ccl_reduce_scatter(inputs, filled, rank, 32, 64, 4, 64, 1)
    else:
        cfg = Config(all_reduce_variant=variant)
        ctx.ccl.all_reduce(d_out, d_in, config=cfg)
        exp = oracle.ccl_all_reduce(inputs, [filled] * W, rank, variant, 32, 64, 4, 64, 1)[rank]
    assert_bits_equal(d_out.cpu(), exp, _lib.last_kernel())


def test_in_place_all_reduce_of_misaligned_rows():
    W, rank, M, N = 4, 2, 37, 131
    ctx = iris.iris(1 << 24, num_ranks=W, rank=rank)
    inputs = [randn_cpu((M, N), 170 + r, torch.bfloat16) for r in range(W)]
    d_in, _ = _stage(ctx, inputs)
    cfg = Config(all_reduce_variant="one_shot")
    ws = ctx.ccl.all_reduce_preamble(ctx.zeros((M, N), dtype=torch.bfloat16), d_in, config=cfg)
    ctx.ccl.all_reduce(d_in, d_in, config=cfg, workspace=ws)
    assert_bits_equal(d_in.cpu(), oracle.ccl_all_reduce(inputs, [inputs[rank]] * W, rank, "one_shot", 32, 64, 4, 64, 1)[rank], "in place")


@pytest.mark.parametrize("op", ["two_shot", "reduce_scatter"])
@pytest.mark.parametrize("W,rank,N", [(8, 0, 4104), (8, 3, 4105), (8, 7, 4104), (3, 1, 2050), (2, 1, 2056)])
def test_large_shares_walked_by_rows(op, W, rank, N):
    """Shares of the block distribution large enough to be walked row by row: they start and end inside a column and
    inside a group of three tile rows, the last group has two; every tile keeps its own order of additions."""
    M, dtype = 4103, torch.bfloat16
    cfg = Config(swizzle_size=3, comm_sms=5)
    ctx = iris.iris(1 << 27, num_ranks=W, rank=rank)
    inputs = [randn_cpu((M, N), 270 + r, dtype) for r in range(W)]
    d_in, d_out = _stage(ctx, inputs, out_fill=3.0)
    filled = torch.full((M, N), 3.0, dtype=dtype)
    if op == "reduce_scatter":
        ctx.ccl.reduce_scatter(d_out, d_in, config=cfg)
        exp = [oracle.ccl_reduce_scatter(inputs, filled, rank, 32, 64, 3, 5, 1) if r == rank else filled for r in range(W)]
    else:
        ctx.ccl.all_reduce(d_out, d_in, config=cfg)
        exp = oracle.ccl_all_reduce(inputs, [filled] * W, rank, "two_shot", 32, 64, 3, 5, 1)
    for r in range(W):
        assert_bits_equal(ctx.peer_view(d_out, r).cpu(), exp[r], f"{_lib.last_kernel()} slot {r}")
