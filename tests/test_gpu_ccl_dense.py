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
    assert "one_shot" in _lib.last_kernel() and "vec1" not in _lib.last_kernel(), _lib.last_kernel()
    exp = torch.zeros((M, N))
    for r in range(W):
        exp += inputs[r].float()
    assert_bits_equal(y.cpu(), exp.to(dtype), f"{W} ranks, {M}x{N}")
    for r in range(W):
        assert_bits_equal(ctx.peer_view(x, r).cpu(), inputs[r], f"input of slot {r}")
        if r != rank:
            assert bool((ctx.peer_view(y, r) == 3.0).all()), f"output of slot {r} was written"
