"""The K loop of the 256x256 tile at its ends: fewer K steps than it keeps in flight, as many, one more, and a partial last step;
in one round of tiles, and in two, where the first step of a workgroup's second tile is fetched ahead."""

import pytest
import torch

import iris_amd as iris
from iris_amd import _lib, ops
from helpers import assert_bits_equal, heap_tensor, oracle, randint_cpu, randn_cpu

pytestmark = pytest.mark.gpu

ONE_ROUND, TWO_ROUNDS = (3072, 3328), (4352, 4352)  # 12 x 13 and 17 x 17 tiles


def _product(A, B, W=1, rank=0, gather_dim=0):
    """all_gather_matmul of A's shards (rows or columns of A, one per rank) and B."""
    shards = list(A.chunk(W, dim=gather_dim))
    ctx = iris.iris(1 << 28, num_ranks=W, rank=rank)
    out_dtype = torch.bfloat16 if A.dtype == torch.float8_e4m3fn else A.dtype
    dA = ctx.zeros(tuple(shards[0].shape), dtype=A.dtype)
    for r in range(W):
        ctx.peer_view(dA, r).copy_(shards[r])
    dB = heap_tensor(ctx, B)
    out = ctx.zeros((A.shape[0], B.shape[1]), dtype=out_dtype)
    cfg = iris.FusedConfig(block_size_m=64, block_size_n=64, block_size_k=8)
    scales = dict(scale_a=1.0, scale_b=1.0) if A.dtype == torch.float8_e4m3fn else {}
    ops.all_gather_matmul(ctx, out, dA, dB, config=cfg, gather_dim=gather_dim, **scales)
    return out.cpu(), _lib.last_kernel()


# K steps are 32 elements of 16 bits, or 64 of e4m3.
@pytest.mark.parametrize("M,N", [ONE_ROUND, TWO_ROUNDS])
@pytest.mark.parametrize("dtype,K", [(torch.bfloat16, k) for k in (8, 32, 40, 64, 96, 104, 128, 160)] +
                         [(torch.float16, 72), (torch.float16, 136)] + [(torch.float8_e4m3fn, k) for k in (16, 64, 128, 192, 208, 256, 320)])
def test_few_k_steps(M, N, dtype, K):
    A, B = randint_cpu((M, K), 300, dtype, -2, 3), randint_cpu((K, N), 301, dtype, -2, 3)
    got, kernel = _product(A, B)
    assert "_256x256x" in kernel and not kernel.endswith("_splitk"), kernel
    out_dtype = torch.bfloat16 if dtype == torch.float8_e4m3fn else dtype
    assert_bits_equal(got, oracle.gemm(A, B, out_dtype), f"{kernel}, K = {K}")


# Gathered along K: sources of one step, of one and a piece, and of three and a piece.
@pytest.mark.parametrize("M,N", [ONE_ROUND, TWO_ROUNDS])
@pytest.mark.parametrize("W,K_local", [(2, 32), (3, 40), (2, 104)])
def test_few_k_steps_of_several_sources(M, N, W, K_local):
    A, B = randint_cpu((M, W * K_local), 302, torch.bfloat16, -2, 3), randint_cpu((W * K_local, N), 303, torch.bfloat16, -2, 3)
    got, kernel = _product(A, B, W, W - 1, gather_dim=1)
    assert "_256x256x" in kernel, kernel
    assert_bits_equal(got, oracle.gemm(A, B, torch.bfloat16), f"{kernel}, {W} sources of {K_local}")


# 16x16x32 products (256x256 tile) and 32x32x16 ones (128x128) of the same rows: random data, no sum exact, 3.4 million results
# rounded to 16 bits; sums that differed in their last bit would round differently in about one of 2^15.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_both_shapes_of_products_give_the_same_bits(dtype):
    M, N, K = 3072, 3328, 2080
    A, B = randn_cpu((M, K), 304, dtype, K ** -0.5), randn_cpu((K, N), 305, dtype)
    big, kernel = _product(A, B)
    assert "_256x256x" in kernel, kernel
    rows, kernel = _product(A[:1024].contiguous(), B)
    assert "_128x128x" in kernel, kernel
    assert_bits_equal(rows, big[:1024], "the same rows on the other tile")
