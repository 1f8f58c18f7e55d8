"""Products of some hundred rows: edges of every tile's rows and columns, one to
a few steps of K, divided and undivided K, the plan's choices."""

import pytest
import torch

from resilient_llm_amd import ops

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


# rows around the tiles of 128, 192 and 256 and their halves, columns around
# those of 128, 256 and 384, steps of K from one to odd and even numbers
SIZES = [(1, 16, 64), (65, 2048, 4096), (127, 136, 128), (129, 272, 192),
         (191, 4112, 448), (193, 1040, 4160), (256, 4080, 320),
         (257, 12304, 256), (385, 8208, 192), (513, 6160, 1088),
         (536, 4096, 14336), (769, 10000, 704), (1025, 4096, 2048),
         (2049, 2064, 640)]


@pytest.mark.parametrize("M,N,K", SIZES)
def test_tile_linear_parts(M, N, K):
    x, w = operands(M, N, K)
    got = torch.ops.rlli.tile_linear_parts(x, w)
    if got.dim() == 3:
        assert got.dtype == torch.float32
        got, half = got.double().sum(0), 0.0
    else:
        half = 2 ** -8                  # half a step of bf16
    # K f32 roundings of sums of size one
    torch.testing.assert_close(got.double(), x.double() @ w.double().T,
                               rtol=half, atol=2 ** -18)


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
    got = torch.ops.rlli.tile_linear_silu(x, w)
    g, u = (x.double() @ w.double().T).chunk(2, 1)
    # a sum's f32 error times the other factor, at most five or so
    torch.testing.assert_close(got.double(),
                               torch.nn.functional.silu(g) * u, rtol=2 ** -8,
                               atol=2 ** -16)


@pytest.mark.parametrize("M,N,K", SIZES)
def test_tile_linear_relu2(M, N, K):
    x, w = operands(M, N, K, 3)
    got = torch.ops.rlli.tile_linear_relu2(x, w)
    want = (x.double() @ w.double().T).clamp(min=0) ** 2
    # the square doubles the product's half step, up to 2^-8 of it, and a sum's
    # f32 error, which it scales by the sum, five or so; then its own half step
    torch.testing.assert_close(got.double(), want, rtol=3 * 2 ** -8,
                               atol=2 ** -14)


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


def test_unaligned_operands_are_refused():
    buf = torch.zeros(300 * 4096 + 1, dtype=torch.bfloat16, device=DEV)
    x = buf[1:1 + 200 * 4096].view(200, 4096)
    w = torch.zeros(4096, 4096, dtype=torch.bfloat16, device=DEV)
    assert not ops.tile_parts_fit(x, w) and not ops.tile_silu_fit(x, w)
    with pytest.raises(RuntimeError, match="multiples of 16"):
        torch.ops.rlli.tile_linear_parts(x, w)
