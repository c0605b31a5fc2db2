"""float32 products on the bf16 matrix pipes (three bf16 pieces per operand): the error against 64 bits, and the operands
whose pieces do not add up to them - infinities, NaN, values next to the largest and below 2^-110 - which are left to
the float32 instructions."""

import pytest
import torch

import iris_amd as iris
from iris_amd import _lib

pytestmark = pytest.mark.gpu

# Output sizes for every tile that splits (on 256 CUs), ragged, and the number of K steps of 32 from one to several.
SHAPES = [(4093, 4095, 31, "128x128"), (4093, 4095, 32, "128x128"), (4093, 4095, 33, "128x128"), (1999, 2877, 32, "64x128"),
          (4093, 4095, 96, "128x128"), (1023, 3969, 333, "128x128"), (1999, 2877, 161, "64x128"), (511, 2879, 1025, "64x64"), (511, 2879, 31, "64x64")]
EPS = 2.0 ** -24


def _product(a, b, b_transposed=False):
    (M, K), N = a.shape, b.shape[1]
    ctx = iris.iris(1 << 27, num_ranks=1, rank=0)
    A, C = ctx.zeros((M, K), dtype=torch.float32), ctx.zeros((M, N), dtype=torch.float32)
    B = ctx.zeros((N, K), dtype=torch.float32).t() if b_transposed else ctx.zeros((K, N), dtype=torch.float32)
    A.copy_(a)
    B.copy_(b)
    ctx.ops.all_gather_matmul(C, A, B, config=iris.FusedConfig(block_size_m=1, block_size_n=64, block_size_k=1), gather_dim=0)
    return C.cpu(), _lib.last_kernel()


@pytest.mark.parametrize("b_transposed", [False, True], ids=["nn", "nt"])
@pytest.mark.parametrize("M,N,K,tile", SHAPES, ids=[f"{s[3]}_k{s[2]}" for s in SHAPES])
def test_error_is_that_of_fp32_sums(M, N, K, tile, b_transposed):
    g = torch.Generator().manual_seed(7)
    a, b = torch.randn((M, K), generator=g), torch.randn((K, N), generator=g)
    b *= torch.exp2(torch.randint(-30, 31, (K, 1), generator=g).float())  # rows of very different sizes
    got, kernel = _product(a, b, b_transposed)
    assert kernel == f"generic_f32_{tile}_" + ("nt" if b_transposed else "nn")
    exact, size = a.double() @ b.double(), a.abs().double() @ b.abs().double()
    # K / 16 slices of six sums rounded to fp32, each by at most 2 eps of what it holds (the matrix pipe cuts
    # off), and 2^-24 of every product left out.
    bound = size * EPS * (2 * 6 * (K // 16 + 1) + 2)
    assert torch.all((got.double() - exact).abs() <= bound), float(((got.double() - exact).abs() / bound).max())
    # Errors of single roundings do not line up: the mean error stays below an eighth of that.
    assert ((got.double() - exact) / bound).abs().mean() < 1 / 8


TILES = [(1023, 3969, "128x128"), (1999, 2877, "64x128"), (511, 2879, "64x64")]


@pytest.mark.parametrize("b_transposed", [False, True], ids=["nn", "nt"])
@pytest.mark.parametrize("M,N,tile", TILES, ids=[t[2] for t in TILES])
def test_every_product_of_pieces_counts(M, N, tile, b_transposed):
    """Single products that fp32 holds: 24 bits of A times one (its pieces all against the first of B; the other
    way round below), and 12 bits of A times 12 bits of B (first and second pieces, all four products)."""
    K, g = 64, torch.Generator().manual_seed(10)
    m, n = torch.arange(M), torch.arange(N)
    a = torch.randint(1 << 23, 1 << 24, (M, K), generator=g).float() * 2.0 ** -23
    one = torch.zeros((K, N))
    one[n % K, n] = 1.0
    got, kernel = _product(a, one, b_transposed)
    assert kernel.startswith(f"generic_f32_{tile}")
    assert torch.equal(got, a[:, n % K])
    a = torch.randint(1 << 11, 1 << 12, (M, K), generator=g).float() * 2.0 ** -11
    one[n % K, n] = torch.randint(1 << 11, 1 << 12, (N,), generator=g).float() * 2.0 ** -11
    got, _ = _product(a, one, b_transposed)
    assert torch.equal(got, a[:, n % K] * one[n % K, n])


@pytest.mark.parametrize("K,limit", [(64, 0.9e-7), (1024, 3.0e-7)])
@pytest.mark.parametrize("M,N,tile", TILES, ids=[t[2] for t in TILES])
def test_error_of_the_sums_in_the_two_norm(M, N, tile, K, limit):
    """Normal operands: 0.50e-7 and 1.9e-7 were measured; with all products of pieces in one sum it is 1.1e-7 and
    4.9e-7, on the float32 instructions 1.4e-7 and 5.7e-7.  The limits lie between the first two."""
    g = torch.Generator().manual_seed(11)
    a, b = torch.randn((M, K), generator=g), torch.randn((K, N), generator=g)
    got, kernel = _product(a, b)
    assert kernel.startswith(f"generic_f32_{tile}")
    exact = a.double() @ b.double()
    assert (got.double() - exact).norm() < limit * exact.norm()


@pytest.mark.parametrize("b_transposed", [False, True], ids=["nn", "nt"])
@pytest.mark.parametrize("M,N,tile", [(4093, 4095, "128x128"), (1999, 2877, "64x128"), (511, 2879, "64x64")])
def test_a_single_product_is_rounded_once(M, N, tile, b_transposed):
    g = torch.Generator().manual_seed(9)
    a, b = torch.randn((M, 1), generator=g), torch.randn((1, N), generator=g)
    got, kernel = _product(a, b, b_transposed)
    assert kernel.startswith(f"generic_f32_{tile}")
    assert torch.equal(got, a * b)


@pytest.mark.parametrize("M,N,K,tile", SHAPES, ids=[f"{s[3]}_k{s[2]}" for s in SHAPES])
def test_operands_that_three_pieces_do_not_hold(M, N, K, tile):
    """One row of A at a time picks single elements of B (powers of two elsewhere zero), so every product is exact in fp32."""
    g = torch.Generator().manual_seed(8)
    b = (torch.randint(1 << 23, 1 << 24, (K, N), generator=g).float() * 2.0 ** -23)  # full 24-bit mantissas
    a = torch.zeros((M, K))
    a[torch.arange(M), torch.arange(M) % K] = 1.0
    expect = b[torch.arange(M) % K]
    got, _ = _product(a, b)
    assert torch.equal(got, expect)  # the pieces add up
    # Just above the limit: the third piece is a subnormal bf16 number, down to its last bit.
    got, _ = _product(a * 2.0 ** 100, b * 2.0 ** -110)
    assert torch.equal(got, expect * 2.0 ** -10)
    # Tiny operands: the last of 24 bits would lie below what bf16 can hold.
    got, _ = _product(a * 2.0 ** 100, b * 2.0 ** -124)
    assert torch.equal(got, expect * 2.0 ** -24)
    # Next to the largest float: the leading piece would round to infinity.
    top = torch.full((K, N), 3.4028234663852886e38)
    top[::2] = -top[::2]
    got, _ = _product(a, top)
    assert torch.equal(got, top[torch.arange(M) % K])
    # Infinities (of both signs, away from zeros of A's row) and NaN stay where they belong.
    odd = b.clone()
    odd[0, 5], odd[0, N - 1], odd[K - 1, 7], odd[K // 2, N // 2] = float("inf"), -float("inf"), float("nan"), float("inf")
    ones = torch.ones((M, K))
    got, _ = _product(ones, odd)
    columns = {5: float("inf"), N - 1: -float("inf"), N // 2: float("inf")}
    for n, value in columns.items():
        assert torch.all(got[:, n] == value), n
    assert torch.all(got[:, 7].isnan())
    finite = torch.ones(N, dtype=torch.bool)
    finite[list(columns) + [7]] = False
    exact = b.double().sum(0)[finite]
    assert torch.all((got[:, finite].double() - exact).abs() <= exact * EPS * (2 * 6 * (K // 16 + 1) + 2))
