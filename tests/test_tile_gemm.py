"""Products of some hundred rows: edges of every tile's rows and columns, one to
a few steps of K, divided and undivided K, the plan's choices, and which
operands are taken."""

import pytest
import torch

from resilient_llm_amd import ops
from resilient_llm_amd.models import llama

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(autouse=True)
def library():
    ops.load_extension(required=True)


def operands(M, N, K, seed=0):
    gen = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=gen).to(torch.bfloat16).to(DEV)
    w = (torch.randn(N, K, generator=gen) * K ** -0.5).to(
        torch.bfloat16).to(DEV)
    return x, w


# what the plan chooses for rows around 128, 192 and 256 and their halves, columns
# around 128, 256 and 384, steps of K from one to odd and even numbers: the tiles
# of 128 x 128, 192 x 128 and 192 x 256 (TILES, by name, are all of them)
SIZES = [(1, 16, 64), (65, 2048, 4096), (127, 136, 128), (129, 272, 192),
         (191, 4112, 448), (193, 1040, 4160), (256, 4080, 320),
         (257, 12304, 256), (385, 8208, 192), (513, 6160, 1088),
         (536, 4096, 14336), (769, 10000, 704), (1025, 4096, 2048),
         (2049, 2064, 640)]


def close_parts(got, x, w):
    if got.dim() == 3:
        assert got.dtype == torch.float32
        got, half = got.double().sum(0), 0.0
    else:
        half = 2 ** -8                  # half a step of bf16
    # K f32 roundings of sums of size one
    torch.testing.assert_close(got.double(), x.double() @ w.double().T,
                               rtol=half, atol=2 ** -18)


def close_silu(got, x, w):
    g, u = (x.double() @ w.double().T).chunk(2, 1)
    # a sum's f32 error times the other factor, at most five or so
    torch.testing.assert_close(got.double(),
                               torch.nn.functional.silu(g) * u, rtol=2 ** -8,
                               atol=2 ** -16)


def close_relu2(got, x, w):
    want = (x.double() @ w.double().T).clamp(min=0) ** 2
    # the square doubles the product's half step, up to 2^-8 of it, and a sum's
    # f32 error, which it scales by the sum, five or so; then its own half step
    torch.testing.assert_close(got.double(), want, rtol=3 * 2 ** -8,
                               atol=2 ** -14)


@pytest.mark.parametrize("M,N,K", SIZES)
def test_tile_linear_parts(M, N, K):
    x, w = operands(M, N, K)
    close_parts(torch.ops.rlli.tile_linear_parts(x, w), x, w)


@pytest.mark.parametrize("M,N,K", SIZES)
def test_tile_linear(M, N, K):
    x, w = operands(M, N, K, 4)
    got = torch.ops.rlli.tile_linear(x, w)
    parts = torch.ops.rlli.tile_linear_parts(x, w)
    if parts.dim() == 3:
        want = parts[0].clone()
        for p in parts[1:]:
            want += p
        parts = want.to(torch.bfloat16)
    assert torch.equal(got, parts)


@pytest.mark.parametrize("M,N,K", SIZES)
def test_tile_linear_silu(M, N, K):
    x, w = operands(M, N - N % 16, K, 1)
    close_silu(torch.ops.rlli.tile_linear_silu(x, w), x, w)


@pytest.mark.parametrize("M,N,K", SIZES)
def test_tile_linear_relu2(M, N, K):
    x, w = operands(M, N, K, 3)
    close_relu2(torch.ops.rlli.tile_linear_relu2(x, w), x, w)


# 64 rows and 128 columns of a tile
TILES = [(2, 1), (2, 2), (2, 3), (3, 1), (3, 2), (3, 3), (4, 1), (4, 2)]


@pytest.mark.parametrize("form", ["whole", "divided", "silu", "relu2"])
@pytest.mark.parametrize("tile", TILES, ids=str)
def test_every_tile(tile, form):
    R, C = 64 * tile[0], 128 * tile[1]
    for M, N, K in [(1, 16, 64), (R // 2 - 1, C // 2 + 16, 128),
                    (R - 1, C - 16, 192), (R, C, 256), (R + 1, C + 16, 320),
                    (3 * R // 2 + 1, 2 * C - 48, 448),
                    (2 * R + 17, 3 * C + 32, 1088)]:
        x, w = operands(M, N, K, M)
        plan = [*tile, min(5, K // 64) if form == "divided" else 1]
        if form == "silu":
            close_silu(torch.ops.rlli.tile_linear_silu(x, w, plan), x, w)
        elif form == "relu2":
            close_relu2(torch.ops.rlli.tile_linear_relu2(x, w, plan), x, w)
        else:
            got = torch.ops.rlli.tile_linear_parts(x, w, plan)
            assert got.shape == ((plan[2], M, N) if plan[2] > 1 else (M, N))
            close_parts(got, x, w)


def test_plans_that_there_are_not():
    x, w = operands(4, 32, 192)
    for plan in ([1, 1, 1], [2, 4, 1], [4, 3, 1], [2, 1, 4], [2, 1, 0],
                 [2, 1], [2, 1, 1 << 33]):
        with pytest.raises(RuntimeError, match="plan"):
            torch.ops.rlli.tile_linear_parts(x, w, plan)
    x, w = operands(4, 32, 1088)
    with pytest.raises(RuntimeError, match="plan"):
        torch.ops.rlli.tile_linear_parts(x, w, [2, 1, 9])
    with pytest.raises(RuntimeError, match="plan"):
        torch.ops.rlli.tile_linear_silu(x, w, [2, 1, 2])


def test_same_bits_in_every_pass():
    x, w = operands(536, 4096, 4096, 2)
    first = torch.ops.rlli.tile_linear_parts(x, w)
    for _ in range(20):
        assert torch.equal(torch.ops.rlli.tile_linear_parts(x, w), first)


@pytest.mark.parametrize("M,N,K", [(64, 64, 96), (64, 60, 64), (64, 24, 0)])
def test_what_does_not_fit(M, N, K):
    x = torch.zeros(M, K, dtype=torch.bfloat16, device=DEV)
    w = torch.zeros(N, K, dtype=torch.bfloat16, device=DEV)
    assert not ops.tile_parts_fit(x, w) and not ops.tile_silu_fit(x, w)
    with pytest.raises(RuntimeError):
        torch.ops.rlli.tile_linear_silu(x, w)


@pytest.mark.parametrize("fit,M,N,K", [
    (ops.tile_parts_fit, 129, 4096, 4096),
    (ops.tile_linear_fit, 129, 4096, 4096),
    (ops.tile_silu_fit, 160, 8192, 2048),
    (ops.tile_relu2_fit, 192, 6144, 2048)])
def test_operands_that_fit(fit, M, N, K):
    """Each condition by itself: what is changed is all that does not fit."""
    def zeros(*shape, dtype=torch.bfloat16):
        return torch.zeros(*shape, dtype=dtype, device=DEV)

    def shifted(t):
        return zeros(t.numel() + 1)[1:].view(t.shape)
    x, w = zeros(M, K), zeros(N, K)
    assert fit(x, w)
    for bad in ((shifted(x), w), (x, shifted(w)),
                (zeros(K, M).T, w), (x, zeros(K, N).T),
                (zeros(M, K + 64)[:, :K], w),
                (x.half(), w.half()), (x.float(), w.float()), (x, w.float()),
                (x.clone().requires_grad_(), w),
                (x, w.clone().requires_grad_()),
                (zeros(M, K + 32), zeros(N, K + 32)), (x, zeros(N + 8, K)),
                (zeros(64, K), w), (zeros(8001, K), w),
                (x[None], w), (x, w[0]), (x.cpu(), w.cpu())):
        assert not fit(*bad)


@pytest.mark.parametrize("M", [64, 65, 128, 129, 160, 161, 191, 192, 256, 257])
def test_products_at_the_limits(M):
    """The ways that the models' products take on either side of a limit."""
    x, w = operands(M, 4096, 4096, 5)
    close_parts(llama._linear(x, w), x, w)
    close_parts(llama._linear_parts(x, w), x, w)
    for N in (8192, 28672):
        x, w = operands(M, N, 2048, 6)
        got = llama._linear_silu(x, w).double()
        g, u = (x.double() @ w.double().T).chunk(2, 1)
        want = torch.nn.functional.silu(g) * u
        # gate and up may be rounded to 16 bits: half a step of either, where
        # silu's slope is up to 1.1
        torch.testing.assert_close(
            got, want, rtol=2 ** -8,
            atol=2 ** -8 * 2.1 * float((g.abs() * u.abs()).max()))
    x, w = operands(M, 6144, 2048, 7)
    close_relu2(llama._linear_relu2(x, w), x, w)


def test_unaligned_operands_are_refused():
    buf = torch.zeros(300 * 4096 + 1, dtype=torch.bfloat16, device=DEV)
    x = buf[1:1 + 200 * 4096].view(200, 4096)
    w = torch.zeros(4096, 4096, dtype=torch.bfloat16, device=DEV)
    assert not ops.tile_parts_fit(x, w) and not ops.tile_silu_fit(x, w)
    with pytest.raises(RuntimeError, match="multiples of 16"):
        torch.ops.rlli.tile_linear_parts(x, w)


@pytest.mark.parametrize("N,K", [(4096, 4096), (6144, 2048), (2048, 6144),
                                 (28672, 4096), (8192, 2048), (260, 3136),
                                 (4080, 1024), (4096, 96)])
def test_the_way_is_that_of_the_rules(N, K):
    w = torch.empty(N, K, dtype=torch.bfloat16, device=DEV)
    for M in (1, 48, 64, 65, 96, 128, 129, 160, 256, 257, 600, 1024, 7000):
        x = torch.empty(M, K, dtype=torch.bfloat16, device=DEV)
        rows = ops.rows_fit(x, w)
        tall = ops._tiles_take(x, w, ops._tall_faster)
        whole, parts, silu, relu2 = (
            ops.product_way(form, M, N, K)
            for form in ("whole", "parts", "silu", "relu2"))
        tile = ops.tile_linear_fit(x, w)
        assert whole == ("tall" if tall else "tile" if tile
                         else "rows" if rows else None)
        assert parts == ("tile" if ops.tile_parts_fit(x, w)
                         else "rows" if rows else None)
        assert silu == ("rows" if rows and N % 16 == 0
                        else "tile" if ops.tile_silu_fit(x, w) else None)
        assert relu2 == ("tall" if tall
                         else "tile" if ops.tile_relu2_fit(x, w)
                         else "rows" if rows and ops.rows_whole(x, w)
                         else None)
