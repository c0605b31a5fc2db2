"""The any-shape kernel at the sizes where its tiles, its K steps and its 16-byte pieces end: every tile, both LDS
layouts of B, every operand type, against the CPU oracle.

Operands are small integers, so products and sums over K are exact in fp32 and the outputs are compared bit for
bit.  They are views into larger buffers that hold NaN around them: whatever the kernel reads beyond an
operand (the rest of a 16-byte piece, rows past the last) must not reach the result.
"""

import pytest
import torch

import iris_amd as iris
from iris_amd import _lib, ops
from helpers import assert_bits_equal, oracle, randint_cpu, randn_cpu, slot_copies, stage_peers

pytestmark = pytest.mark.gpu

FP8 = torch.float8_e4m3fn


def _view(ctx, value, transposed=False, slot=None):
    """`value` as the top left corner of a heap buffer of NaNs (stored transposed: a view without unit column stride)."""
    v = value.t() if transposed else value
    rows, cols = v.shape
    wide = ctx.zeros((rows + 3, cols + 3), dtype=v.dtype)
    wide.copy_(torch.full((rows + 3, cols + 3), float("nan")).to(v.dtype))
    wide[:rows, :cols].copy_(v)
    view = wide[:rows, :cols]
    return view.t() if transposed else view


def _ints(shape, seed, dtype):
    return randint_cpu(shape, seed, torch.float32, -3, 4).to(dtype)


# Tile the host picks on 256 CUs -> output size; columns end 1, 4 or 7 short of (or past) a piece, rows past a tile.
TILES = {"256x256": (4095, 4093), "128x128": (2303, 3137), "64x128": (1030, 3137), "64x64": (641, 2369), "32x32": (67, 295)}
TILES_F32 = {"256x256": "128x128", "64x128": "128x128"}  # where float32 takes another tile


@pytest.mark.parametrize("b_transposed", [False, True], ids=["nn", "nt"])
@pytest.mark.parametrize("tile", sorted(TILES))
@pytest.mark.parametrize("dtype,K", [(torch.bfloat16, 129), (torch.float16, 63), (FP8, 257), (torch.float32, 65)],
                         ids=["bf16", "f16", "fp8", "f32"])
def test_every_tile_and_type(dtype, K, tile, b_transposed):
    M, N = TILES[tile]
    W, rank = 2, 1
    out_dtype = torch.bfloat16 if dtype == FP8 else dtype
    ctx = iris.iris(1 << 28, num_ranks=W, rank=rank)
    A, B = _ints((M, K), 1, dtype), _ints((K, N), 2, dtype)
    peers = [randn_cpu((M, N), 30 + r, out_dtype) for r in range(W)]
    cfg = iris.FusedConfig(block_size_m=64, block_size_n=24, block_size_k=16, all_reduce_variant="one_shot")
    dA, dB, dC = _view(ctx, A), _view(ctx, B, b_transposed), ctx.zeros((M, N), dtype=out_dtype)
    ws = ops.matmul_all_reduce_preamble(ctx, dC, dA, dB, config=cfg)
    stage_peers(ctx, ws, peers)
    ops.matmul_all_reduce(ctx, dC, dA, dB, config=cfg, workspace=ws)
    kernel = _lib.last_kernel()
    expected = TILES_F32.get(tile, tile) if dtype == torch.float32 else tile
    assert kernel.startswith("generic_") and kernel.endswith(f"_{expected}_" + ("nt" if b_transposed else "nn")), kernel
    exp = oracle.matmul_all_reduce(A, B, peers, rank, W, 64, 24, "one_shot", out_dtype=out_dtype)
    assert_bits_equal(ws.aux_buffer.cpu(), exp["aux"], f"{kernel}: aux")
    assert_bits_equal(dC.cpu(), exp["C"][rank], f"{kernel}: C")
    assert torch.all(ws.locks.cpu() == 1), kernel


# N below one 16-byte piece, a tile of fewer columns than a piece, K below a piece, one row.
@pytest.mark.parametrize("M,N,K", [(1, 5, 3), (3, 33, 8), (70, 129, 511), (1, 2881, 1001), (130, 7, 64)])
@pytest.mark.parametrize("variant", ["one_shot", "two_shot", "atomic"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
def test_narrow_outputs_and_owners_inside_pieces(dtype, variant, M, N, K):
    """Flag tiles of 5 columns: pieces of several owners.  The atomic variant adds aligned dwords of rows that
    start in the middle of one."""
    W, rank = 4, 2
    ctx = iris.iris(1 << 24, num_ranks=W, rank=rank)
    A, B = _ints((M, K), 3, dtype), _ints((K, N), 4, dtype)
    peers = [_ints((M, N), 50 + r, dtype) for r in range(W)]
    cfg = iris.FusedConfig(block_size_m=1, block_size_n=5, block_size_k=1, all_reduce_variant=variant)
    dA, dB, dC = _view(ctx, A), _view(ctx, B), ctx.zeros((M, N), dtype=dtype)
    ws = ops.matmul_all_reduce_preamble(ctx, dC, dA, dB, config=cfg)
    for r in range(W):  # (a fresh heap holds whatever was there)
        if variant == "atomic":
            ctx.peer_view(dC, r).copy_(peers[r])
        else:
            ctx.peer_view(dC, r).zero_()
    if variant != "atomic":
        stage_peers(ctx, ws, peers)
    ops.matmul_all_reduce(ctx, dC, dA, dB, config=cfg, workspace=ws, kernel_path="generic")
    exp = oracle.matmul_all_reduce(A, B, peers, rank, W, 1, 5, variant)
    for r, got in enumerate(slot_copies(ctx, dC)):
        assert_bits_equal(got, exp["C"][r], f"{_lib.last_kernel()} slot {r}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, FP8, torch.float32], ids=["bf16", "fp8", "f32"])
@pytest.mark.parametrize("gather_dim,W,M,Kl,N", [(1, 3, 131, 67, 261), (1, 8, 40, 129, 2051), (0, 3, 43, 131, 517), (0, 5, 1, 70, 33)])
def test_gathered_transposed_and_strided_operands(dtype, gather_dim, W, M, Kl, N):
    """Odd shares of K per slot, tiles that span several slots' rows; A handed over transposed, B without a unit
    stride, C with strided columns, a row bias."""
    rank = W - 1
    out_dtype = torch.bfloat16 if dtype == FP8 else dtype
    ctx = iris.iris(1 << 27, num_ranks=W, rank=rank)
    shards = [_ints((M, Kl), 60 + r, dtype) for r in range(W)]
    K, rows = (W * Kl, M) if gather_dim == 1 else (Kl, W * M)
    B, bias = _ints((K, N), 70, dtype), randint_cpu((rows,), 71, out_dtype, -8, 9)
    cfg = iris.FusedConfig(block_size_m=1, block_size_n=16, block_size_k=1)
    exp = oracle.all_gather_matmul(shards, B, bias=bias, gather_dim=gather_dim, out_dtype=out_dtype)
    for a_t, b_strided, c_strided in ((False, False, True), (True, False, False), (False, True, False)):
        buf = ctx.zeros((Kl, M) if a_t else (M, Kl), dtype=dtype)
        for r in range(W):
            ctx.peer_view(buf, r).copy_(shards[r].t() if a_t else shards[r])
        dA = buf.t() if a_t else buf
        dB = ctx.zeros((K, 2 * N), dtype=dtype)[:, ::2] if b_strided else ctx.zeros((K, N), dtype=dtype)
        dB.copy_(B)
        out = ctx.zeros((rows, 2 * N), dtype=out_dtype)[:, ::2] if c_strided else ctx.zeros((rows, N), dtype=out_dtype)
        ops.all_gather_matmul(ctx, out, dA, dB, bias=bias.cuda(), config=cfg, gather_dim=gather_dim)
        kernel = _lib.last_kernel()
        assert kernel.startswith("generic"), kernel
        assert_bits_equal(out.cpu(), exp, f"{kernel} a_t={a_t} b_strided={b_strided} c_strided={c_strided}")


# Bits that no arithmetic may pass over: signalling and quiet NaNs with a payload, subnormals, -0, infinity.
PATTERNS = {torch.bfloat16: [0x7f81, 0xffa1, 0x7fc3, 0x0001, 0x807f, 0x8000, 0x7f80], torch.float16: [0x7c01, 0xfd01, 0x7e03, 0x0001, 0x83ff, 0x8000, 0x7c00]}


# Columns that start and end in the middle of a dword, at either end, rows one after the other without a gap.
@pytest.mark.parametrize("M,N,first,stride", [(67, 294, 1, 304), (67, 295, 1, 303), (67, 295, 0, 304), (5, 1, 3, 9), (641, 2370, 1, 2400), (67, 295, 0, 295)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
def test_atomic_leaves_what_lies_next_to_c(dtype, M, N, first, stride):
    W, rank, K = 3, 1, 24
    ctx = iris.iris(1 << 24, num_ranks=W, rank=rank)
    A, B = _ints((M, K), 5, dtype), _ints((K, N), 6, dtype)
    size, begin = M * stride + 8, 1  # (with a row stride of N the elements in front of and behind all of C)
    flat = ctx.zeros((size,), dtype=dtype)
    C = flat[begin:begin + M * stride].view(M, stride)[:, first:first + N]
    bits = torch.tensor(PATTERNS[dtype], dtype=torch.int32).to(torch.int16)[torch.arange(size) % 7]
    cfg = iris.FusedConfig(block_size_m=1, block_size_n=1, block_size_k=1, all_reduce_variant="atomic")
    dA, dB = _view(ctx, A), _view(ctx, B)
    ws = ops.matmul_all_reduce_preamble(ctx, C, dA, dB, config=cfg)
    exp = bits.clone()
    exp[begin:begin + M * stride].view(M, stride)[:, first:first + N] = (oracle.gemm(A, B).float() + 1).to(dtype).view(torch.int16)
    for r in range(W):
        ctx.peer_view(flat, r).view(torch.int16).copy_(bits)
        ctx.peer_view(flat, r)[begin:begin + M * stride].view(M, stride)[:, first:first + N].fill_(1.0)
    ops.matmul_all_reduce(ctx, C, dA, dB, config=cfg, workspace=ws, kernel_path="generic")
    for r, got in enumerate(slot_copies(ctx, flat)):
        assert torch.equal(got.view(torch.int16), exp), f"{_lib.last_kernel()} slot {r}"
