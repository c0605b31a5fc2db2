"""A workspace handed back to the operator that used it: the second call runs no preamble and must still leave what a
call with one leaves - own tiles reduced, every other tile of C zero - on each kernel family."""

import ctypes
import subprocess
import sys

import pytest
import torch

import iris_amd as iris
from iris_amd import _lib, ops
from iris_amd.ccl import Config
from helpers import assert_bits_equal, heap_tensor, oracle, randint_cpu, randn_cpu, stage_peers

pytestmark = pytest.mark.gpu


# 32x32 kernel, 64x64 and 256x256 tiles, the any-shape kernel with whole and with ragged pieces.
@pytest.mark.parametrize("M,N,K,dtype,kernel", [
    (96, 264, 72, torch.bfloat16, "mfma_bf16_32x32"), (640, 1024, 96, torch.float16, "mfma_f16_64x64"), (3072, 3080, 80, torch.bfloat16, "mfma_bf16_256x256"),
    (130, 132, 40, torch.float32, "generic_f32"), (131, 267, 70, torch.float16, "generic_f16")])
@pytest.mark.parametrize("op", ["one_shot", "two_shot", "atomic", "reduce_scatter"])
def test_second_call_equals_first(op, M, N, K, dtype, kernel):
    W, rank = 4, 2
    ctx = iris.iris(1 << 27, num_ranks=W, rank=rank)
    B = randint_cpu((K, N), 1, dtype)
    peers = [randn_cpu((M, N), 20 + r, dtype) for r in range(W)]
    dA, dB, dC = ctx.zeros((M, K), dtype=dtype), heap_tensor(ctx, B), ctx.zeros((M, N), dtype=dtype)
    variant = "two_shot" if op == "reduce_scatter" else op
    cfg = iris.FusedConfig(block_size_m=32, block_size_n=24, block_size_k=16, all_reduce_variant=variant)
    preamble = ops.matmul_reduce_scatter_preamble if op == "reduce_scatter" else ops.matmul_all_reduce_preamble
    call = ops.matmul_reduce_scatter if op == "reduce_scatter" else ops.matmul_all_reduce
    ws = preamble(ctx, dC, dA, dB, cfg)
    if op != "atomic":
        stage_peers(ctx, ws, peers)
    side = torch.cuda.Stream()
    for turn in range(4):
        A = randint_cpu((M, K), 40 + turn, dtype)
        dA.copy_(A)
        if turn:  # (the first call relies on the preamble's zeros)
            dC.fill_(float("nan"))  # nothing of what C holds may survive
        torch.cuda.synchronize()
        with torch.cuda.stream(side if turn == 2 else torch.cuda.current_stream()):  # turns 2 and 3: another stream than before
            ws = call(ctx, dC, dA, dB, async_op=True, config=cfg, workspace=ws)
        torch.cuda.synchronize()
        assert _lib.last_kernel().startswith(kernel), _lib.last_kernel()
        if op == "atomic":
            exp = oracle.gemm(A, B)  # added to a zeroed C
        elif op == "reduce_scatter":
            exp = oracle.matmul_reduce_scatter(A, B, peers, rank, W, 32, 24)["C"][rank]
        else:
            exp = oracle.matmul_all_reduce(A, B, peers, rank, W, 32, 24, variant)["C"][rank]
        assert_bits_equal(dC.cpu() + 0, exp + 0, f"{op} turn {turn}")  # (+ 0: zeros of one sign)
        ctx.check_status()


@pytest.mark.parametrize("variant", ["one_shot", "atomic"])
def test_second_collective_equals_first(variant):
    W, rank, M, N, dtype = 4, 1, 70, 264, torch.bfloat16
    ctx = iris.iris(1 << 24, num_ranks=W, rank=rank)
    x, y = ctx.zeros((M, N), dtype=dtype), ctx.zeros((M, N), dtype=dtype)
    cfg = Config(all_reduce_variant=variant)
    ws = ctx.ccl.all_reduce_preamble(y, x, config=cfg)
    for turn in range(3):
        inputs = [randint_cpu((M, N), 10 * turn + r, dtype) for r in range(W)]
        for r in range(W):
            ctx.peer_view(x, r).copy_(inputs[r])
        if turn:
            y.fill_(float("nan"))
        ws = ctx.ccl.all_reduce(y, x, async_op=True, config=cfg, workspace=ws)
        exp = sum(i.float() for i in inputs).to(dtype) if variant == "one_shot" else inputs[rank]
        assert_bits_equal(y.cpu() + 0, exp + 0, f"turn {turn}")


def test_calls_that_are_not_in_order_reach_the_python_checks():
    """The native call path takes calls that are plainly in order and must leave every other one to the wrapper's
    checks and messages, also on a workspace it has used."""
    W, M, N, K, dtype = 2, 64, 128, 64, torch.bfloat16
    ctx = iris.iris(1 << 24, num_ranks=W, rank=0)
    A, B, C = ctx.zeros((M, K), dtype=dtype), ctx.zeros((K, N), dtype=dtype), ctx.zeros((M, N), dtype=dtype)
    cfg = iris.FusedConfig(block_size_m=32, block_size_n=32, block_size_k=32, all_reduce_variant="one_shot")
    ws = ops.matmul_all_reduce_preamble(ctx, C, A, B, config=cfg)
    stage_peers(ctx, ws, [C] * W)
    for _ in range(2):
        ws = ctx.ops.matmul_all_reduce(C, A, B, config=cfg, workspace=ws)
    with pytest.raises(ValueError, match="Incompatible matrix dimensions"):
        ctx.ops.matmul_all_reduce(C, A, B[:32], config=cfg, workspace=ws)
    with pytest.raises(ValueError, match="same dtype"):
        ctx.ops.matmul_all_reduce(C, A, B.half(), config=cfg, workspace=ws)
    with pytest.raises(ValueError, match="scale_a"):
        ctx.ops.matmul_all_reduce(C, A, B, config=cfg, workspace=ws, scale_a=1.0)
    with pytest.raises(ValueError, match="kernel path"):
        ctx.ops.matmul_all_reduce(C, A, B, config=cfg, workspace=ws, kernel_path="fast")
    with pytest.raises(RuntimeError, match="is on cpu"):
        ctx.ops.matmul_all_reduce(C, A, B.cpu(), config=cfg, workspace=ws)
    with pytest.raises(AssertionError, match="too small for block_size_m"):
        ctx.ops.matmul_all_reduce(C, A, B, config=iris.FusedConfig(all_reduce_variant="one_shot"), workspace=ws)
    with pytest.raises(RuntimeError, match="symmetric heap"):
        ctx.ops.all_gather_matmul(C, torch.zeros((M, K // W), dtype=dtype, device="cuda"), B, config=cfg)
    with pytest.raises(RuntimeError, match="symmetric heap"):
        ctx.ops.matmul_all_gather(torch.zeros((W * M, N), dtype=dtype, device="cuda"), A, B, config=cfg)
    with pytest.raises(RuntimeError, match="symmetric heap"):
        ctx.ccl.reduce_scatter(C, torch.zeros((M, N), dtype=dtype, device="cuda"))
    ctx._status[0] = _lib.STATUS_SPIN_TIMEOUT  # as a kernel of an earlier call would leave it
    with pytest.raises(RuntimeError, match="gave up waiting"):
        ctx.ops.matmul_all_reduce(C, A, B, config=cfg, workspace=ws)
    ws = ctx.ops.matmul_all_reduce(C, A, B, config=cfg, workspace=ws)
    assert torch.all(C == 0)


def test_tensors_without_memory_are_refused():
    """Inside vmap a batched operand has no address: an exception, raised where Python can take it."""
    W, M, N, K, dtype = 2, 64, 128, 64, torch.bfloat16
    ctx = iris.iris(1 << 24, num_ranks=W, rank=0)
    A, B, C = ctx.zeros((M, K), dtype=dtype), ctx.zeros((K, N), dtype=dtype), ctx.zeros((M, N), dtype=dtype)
    wide, Bs = ctx.zeros((W * M, N), dtype=dtype), torch.zeros((3, K, N), dtype=dtype, device="cuda")
    cfg = iris.FusedConfig(block_size_m=32, block_size_n=32, block_size_k=32, all_reduce_variant="one_shot")
    ws = ops.matmul_all_reduce_preamble(ctx, C, A, B, config=cfg)
    rs = ops.matmul_reduce_scatter_preamble(ctx, C, A, B, config=cfg)
    rs.stream = torch.cuda.current_stream().cuda_stream
    ccl = ctx.ccl.all_reduce_preamble(C, wide[:K], config=Config(all_reduce_variant="one_shot"))
    calls = [
        lambda b: ctx.ops.matmul_all_reduce(C, A, b, config=cfg, workspace=ws),
        lambda b: ctx.ops.matmul_reduce_scatter(C, A, b, config=cfg, workspace=rs, sum_peers=False),
        lambda b: ctx.ops.all_gather_matmul(wide, A, b, config=cfg, gather_dim=0),
        lambda b: ctx.ops.matmul_all_gather(wide, A, b, config=cfg),
        lambda b: ctx.ccl.all_reduce(b, wide[:K], config=Config(all_reduce_variant="one_shot"), workspace=ccl),
        lambda b: ctx.ccl.reduce_scatter(b, wide[:K]),
    ]
    for call in calls:
        with pytest.raises(RuntimeError, match="data pointer|storage"):
            torch.vmap(lambda b: (call(b), b)[1])(Bs)


_FAILING = """
int calls = 0;
int iris_hip_matmul_all_reduce() { return ++calls, 98; }
int iris_hip_matmul_reduce_scatter() { return ++calls, 98; }
int iris_hip_all_gather_matmul() { return ++calls, 98; }
int iris_hip_matmul_all_gather() { return ++calls, 98; }
int iris_hip_all_reduce() { return ++calls, 98; }
int iris_hip_reduce_scatter() { return ++calls, 98; }
int iris_hip_stream_capturing() { return 0; }
"""


def test_a_failed_launch_is_reported_and_not_repeated(tmp_path):
    """Entry points that return an error behind a launch that went out (as an earlier call's error does): one call, one
    exception, and the workspace as it was."""
    W, M, N, K, dtype = 2, 64, 128, 64, torch.bfloat16
    ctx = iris.iris(1 << 24, num_ranks=W, rank=0)
    A, B, C = ctx.zeros((M, K), dtype=dtype), ctx.zeros((K, N), dtype=dtype), ctx.zeros((M, N), dtype=dtype)
    wide = ctx.zeros((W * M, N), dtype=dtype)
    cfg = iris.FusedConfig(block_size_m=32, block_size_n=32, block_size_k=32, all_reduce_variant="atomic")
    one_shot = Config(all_reduce_variant="one_shot")
    ws = ops.matmul_all_reduce_preamble(ctx, C, A, B, config=cfg)
    rs = ctx.ops.matmul_reduce_scatter(C, A, B, config=cfg, sum_peers=False)
    ccl = ctx.ccl.all_reduce_preamble(C, wide[:M], config=one_shot)
    calls = [
        lambda: ctx.ops.matmul_all_reduce(C, A, B, config=cfg, workspace=ws),
        lambda: ctx.ops.matmul_reduce_scatter(C, A, B, config=cfg, workspace=rs, sum_peers=False),
        lambda: ctx.ops.all_gather_matmul(wide, A, B, config=cfg, gather_dim=0),
        lambda: ctx.ops.matmul_all_gather(wide, A, B, config=cfg),
        lambda: ctx.ccl.all_reduce(C, wide[:M], config=one_shot, workspace=ccl),
        lambda: ctx.ccl.reduce_scatter(C, wide[:M]),
    ]
    (tmp_path / "failing.c").write_text(_FAILING)
    path = str(tmp_path / "failing.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", path, str(tmp_path / "failing.c")], check=True)
    count = ctypes.c_int.in_dll(ctypes.CDLL(path), "calls")
    _lib.launcher().load(path)
    try:
        for i, call in enumerate(calls):
            with pytest.raises(RuntimeError, match="HIP error code 98"):
                call()
            assert count.value == i + 1, f"call {i}: entry points were called {count.value - i} times"
    finally:
        _lib.launcher().load(_lib.LIBRARY_PATH)
    assert ws.prepared and ws.stream is None and ccl.prepared and ccl.stream is None
    for call in calls:
        call()


class _Preamble(Exception):
    pass


@pytest.mark.parametrize("op", ["one_shot", "atomic", "reduce_scatter", "ccl"])
@pytest.mark.parametrize("wrapper", [False, True], ids=["native", "wrapper"])
def test_launches_in_graphs_and_the_preamble(op, wrapper, monkeypatch):
    """A used workspace is not taken as it is while a graph is recorded (the preamble, which cannot be recorded, is asked
    for), nor ever again once a launch that uses it is part of a graph, whose replays run on any stream."""
    W, M, N, K, dtype = 2, 64, 128, 64, torch.bfloat16
    ctx = iris.iris(1 << 24, num_ranks=W, rank=0)
    A, B, C, x = (ctx.zeros(s, dtype=dtype) for s in ((M, K), (K, N), (M, N), (M, N)))
    cfg = iris.FusedConfig(block_size_m=32, block_size_n=32, block_size_k=32, all_reduce_variant="two_shot" if op == "reduce_scatter" else op)
    ccl_cfg = Config(all_reduce_variant="one_shot")
    if op == "ccl":
        module, name = sys.modules["iris_amd.ccl.all_reduce"], "all_reduce_preamble"
        ctx.peer_view(x, 1).zero_()  # (a heap's memory is as it was found; zeros() clears the own slot)
        ws = ctx.ccl.all_reduce_preamble(C, x, config=ccl_cfg)
        call = lambda: ctx.ccl.all_reduce(C, x, async_op=True, config=ccl_cfg, workspace=ws)
    elif op == "reduce_scatter":
        module, name = sys.modules["iris_amd.ops.matmul_reduce_scatter"], "matmul_reduce_scatter_preamble"
        ws = ops.matmul_reduce_scatter_preamble(ctx, C, A, B, config=cfg)
        call = lambda: ctx.ops.matmul_reduce_scatter(C, A, B, async_op=True, config=cfg, workspace=ws, sum_peers=False)
    else:
        module, name = sys.modules["iris_amd.ops.matmul_all_reduce"], "matmul_all_reduce_preamble"
        ws = ops.matmul_all_reduce_preamble(ctx, C, A, B, config=cfg)
        call = lambda: ctx.ops.matmul_all_reduce(C, A, B, async_op=True, config=cfg, workspace=ws)
        if op == "one_shot":
            stage_peers(ctx, ws, [C] * W)
    preamble, asked = getattr(module, name), []

    def refuse(*args, **kwargs):
        asked.append(1)
        raise _Preamble

    if wrapper:
        monkeypatch.setattr(module, "native", lambda shmem: None)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
        call()
        torch.cuda.synchronize()
        monkeypatch.setattr(module, name, refuse)
        call()  # as it is, without the preamble (the reduce-scatter's first call ran it)
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=side):
            with pytest.raises(_Preamble):
                call()
            if op != "reduce_scatter":  # (which has no launch without a preamble before it)
                ws.prepared = True
                call()
        assert len(asked) == 1
        if op == "reduce_scatter":
            return
        for _ in range(2):
            graph.replay()
            torch.cuda.synchronize()
            ctx.check_status()
            assert torch.all(C == 0)
        with pytest.raises(_Preamble):
            call()
        monkeypatch.setattr(module, name, preamble)
        call()  # with the preamble, and the next one too
        monkeypatch.setattr(module, name, refuse)
        with pytest.raises(_Preamble):
            call()
        torch.cuda.synchronize()


@pytest.mark.parametrize("variant,W,rank", [("one_shot", 4, 1), ("two_shot", 1, 0)])
def test_second_call_of_a_split_launch(variant, W, rank):
    """The last round's tiles split between workgroups, flag tiles higher than the workgroups' (their arrivals are counted
    in the flag): calls that find their own flags up give what the oracle gives."""
    M, N, K, dtype = 5120, 3840, 200, torch.bfloat16
    ctx = iris.iris(1 << 29, num_ranks=W, rank=rank)
    B = randint_cpu((K, N), 6, dtype)
    peers = [randn_cpu((M, N), 40 + r, dtype) for r in range(W)]
    cfg = iris.FusedConfig(block_size_m=384, block_size_n=64, block_size_k=32, all_reduce_variant=variant)
    dA, dB, dC = ctx.zeros((M, K), dtype=dtype), heap_tensor(ctx, B), ctx.zeros((M, N), dtype=dtype)
    ws = ops.matmul_all_reduce_preamble(ctx, dC, dA, dB, config=cfg)
    stage_peers(ctx, ws, peers)
    _lib.library().iris_hip_set_split_tiles(1)
    try:
        for turn in range(3):
            A = randint_cpu((M, K), 5 + turn, dtype)
            dA.copy_(A)
            if turn:
                dC.fill_(float("nan"))
            ws = ops.matmul_all_reduce(ctx, dC, dA, dB, config=cfg, workspace=ws)
            assert _lib.last_kernel().endswith("_splitk"), _lib.last_kernel()
            exp = oracle.matmul_all_reduce(A, B, peers, rank, W, 384, 64, variant, "fp32")
            assert torch.equal(ws.locks.cpu(), torch.from_numpy(exp["locks"])), "flags"
            assert_bits_equal(dC.cpu(), exp["C"][rank], f"turn {turn}")
    finally:
        _lib.library().iris_hip_set_split_tiles(-1)
