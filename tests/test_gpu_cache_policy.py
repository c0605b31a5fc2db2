"""The ways the peers' tiles are read (through the caches or past them, by the bytes a launch reads) and aux is written (rows of
whole 128-byte lines, or not): both sides of each line, tiled and any-shape kernels, against the CPU oracle, bit for bit."""

import pytest
import torch

import iris_amd as iris
from iris_amd import ops
from helpers import assert_bits_equal, heap_tensor, oracle, randint_cpu, randn_cpu, slot_copies, stage_peers

pytestmark = pytest.mark.gpu

# Read from seven peers: one-shot 7 MN elements, with owners 7/8 MN; the line lies at 32 MiB.
CASES = [
    (torch.bfloat16, "one_shot", 1008, 2368, 32),   # 33.4 MB, just below
    (torch.bfloat16, "one_shot", 1024, 2368, 32),   # 33.9 MB, just above; rows of whole lines
    (torch.float16, "one_shot", 1024, 2376, 32),    # above, rows that are not
    (torch.float16, "two_shot", 4096, 4736, 24),    # 33.9 MB, above
    (torch.bfloat16, "two_shot", 4032, 4744, 24),   # 33.5 MB, below, rows that are not whole lines
    (torch.float32, "one_shot", 512, 2400, 16),     # any-shape kernel, above
    (torch.bfloat16, "one_shot", 1023, 2377, 17),   # any-shape kernel, above, odd rows
    (torch.bfloat16, "one_shot", 511, 2377, 17),    # ... below
]


@pytest.mark.parametrize("dtype,variant,M,N,K", CASES)
def test_both_ways_agree_with_the_oracle(dtype, variant, M, N, K):
    W, rank = 8, 3
    ctx = iris.iris(1 << 27, num_ranks=W, rank=rank)
    A, B = randint_cpu((M, K), 1, dtype), randint_cpu((K, N), 2, dtype)
    peers = [randn_cpu((M, N), 20 + r, dtype) for r in range(W)]
    cfg = iris.FusedConfig(block_size_m=128, block_size_n=64, block_size_k=16, all_reduce_variant=variant)
    dA, dB, dC = heap_tensor(ctx, A), heap_tensor(ctx, B), ctx.zeros((M, N), dtype=dtype)
    ws = ops.matmul_all_reduce_preamble(ctx, dC, dA, dB, config=cfg)
    stage_peers(ctx, ws, peers)
    ops.matmul_all_reduce(ctx, dC, dA, dB, config=cfg, workspace=ws)
    exp = oracle.matmul_all_reduce(A, B, peers, rank, W, 128, 64, variant)
    assert_bits_equal(ws.aux_buffer.cpu(), exp["aux"], "aux")
    assert torch.equal(ws.locks.cpu(), torch.from_numpy(exp["locks"]))
    if variant == "one_shot":
        assert_bits_equal(dC.cpu(), exp["C"][rank], "C")
    else:
        for r, got in enumerate(slot_copies(ctx, dC)):
            assert_bits_equal(got, exp["C"][r], f"C in slot {r}")
