"""Products of few rows: edges of row tiles, weight panels, the ring of K
steps and the division of K; a row's result is the same in any batch of up to
64 rows, and in any larger one."""

import pytest
import torch

from resilient_llm_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ROWS = [1, 15, 16, 17, 32, 33, 48, 49, 64, 65, 96, 97]


def operands(N, K, seed=0):
    gen = torch.Generator().manual_seed(seed)
    x = torch.randn(128, K, generator=gen).to(torch.bfloat16).to(DEV)
    w = torch.randn(N, K, generator=gen).to(torch.bfloat16).to(DEV)
    return x, w


def close(got, want, size, rtol=2 ** -8):
    # half a step of bf16 for the result, K f32 roundings of sums of ``size``
    torch.testing.assert_close(got.double(), want, rtol=rtol,
                               atol=float(size) * 2 ** -20)


@pytest.mark.parametrize("N,K", [
    (4, 64), (60, 64), (64, 128), (68, 192), (6160, 320), (8196, 448),
    (16448, 64), (25540, 192), (25664, 704), (1536, 4096),
    # panels of 8 to 32 rows with K divided among a workgroup's waves:
    # fewer steps than waves, some waves one step more, around the lines
    # between the kernels
    (4096, 192), (4100, 320), (8188, 704), (4092, 3072), (2048, 3136),
    (508, 8192), (516, 8192), (4112, 4096), (4100, 4160)])
def test_rows_linear(N, K):
    x, w = operands(N, K)
    whole = ops.rows_linear(x, w)
    close(whole, x.double() @ w.double().T, K ** 0.5)
    few = ops.rows_linear(x[:64].contiguous(), w)
    close(few, x[:64].double() @ w.double().T, K ** 0.5)
    for m in ROWS:
        assert torch.equal(ops.rows_linear(x[:m].contiguous(), w),
                           (few if m <= 64 else whole)[:m])
    if torch.ops.rlli.rows_whole_ok(64, N, K):
        got = torch.ops.rlli.rows_linear_relu2(x[:64].contiguous(), w)
        y = x[:64].double() @ w.double().T
        # the square doubles a sum's relative error and scales it by the sum
        close(got, y.clamp(min=0) ** 2, 8 * K)
    parts = torch.ops.rlli.rows_linear_parts(x, w)
    if parts.dim() == 3:
        s = parts[0].clone()
        for p in parts[1:]:
            s += p
        assert torch.equal(s.to(torch.bfloat16), whole)


@pytest.mark.parametrize("N", [
    # a workgroup's 8, 16, 24 or 32 rows of w: the lines between them, a last one
    # with few rows, a half tile that is not there
    4, 2044, 2048, 2052, 4092, 4096, 4104, 6120, 6132, 6144, 6148, 8184])
def test_rows_of_a_workgroup(N):
    x, w = operands(N, 576, N)
    want = x[:64].double() @ w.double().T
    few = ops.rows_linear(x[:64].contiguous(), w)
    close(few, want, 24)
    for m in (1, 16, 17, 32, 33):
        assert torch.equal(ops.rows_linear(x[:m].contiguous(), w), few[:m])


@pytest.mark.parametrize("inter,K", [(8, 64), (72, 128), (5152, 64),
                                     (12744, 192), (12800, 448)])
def test_rows_linear_silu(inter, K):
    x, w = operands(2 * inter, K, 1)
    w *= K ** -0.5
    whole = torch.ops.rlli.rows_linear_silu(x, w)
    g, u = (x.double() @ w.double().T).chunk(2, 1)
    # a sum's f32 error times the other factor, both of size one; few pairs
    # take the product in 16 bits, whose half steps grow with 1 + |gate|
    close(whole, torch.nn.functional.silu(g) * u, 8.0,
          2 ** -8 if inter > 5000 else 8 * 2 ** -8)
    for m in ROWS:
        assert torch.equal(
            torch.ops.rlli.rows_linear_silu(x[:m].contiguous(), w), whole[:m])


@pytest.mark.parametrize("M,N,K", [(129, 64, 64), (1, 64, 96), (1, 6, 64)])
def test_what_does_not_fit(M, N, K):
    x = torch.zeros(M, K, dtype=torch.bfloat16, device=DEV)
    w = torch.zeros(N, K, dtype=torch.bfloat16, device=DEV)
    assert not ops.rows_fit(x, w)
    with pytest.raises(RuntimeError):
        ops.rows_linear(x, w)


@pytest.mark.parametrize("n,rows,dim", [(1, 1, 8), (2, 3, 520), (5, 64, 4096),
                                        (8, 2, 8192)])
def test_norm_of_parts(n, rows, dim):
    gen = torch.Generator().manual_seed(dim)
    parts = torch.randn(n, rows, dim, generator=gen).to(DEV)
    res = torch.randn(rows, dim, generator=gen).to(torch.bfloat16).to(DEV)
    w = torch.randn(dim, generator=gen).to(torch.bfloat16).to(DEV)
    want = (parts.double().sum(0) + res.double())
    got = ops.rmsnorm_residual_(parts, res, w, 1e-5)
    # the f32 sum's rounding may move a result to the next bf16 number
    torch.testing.assert_close(res.double(), want, rtol=2 ** -8,
                               atol=n * 2 ** -20)
    r = res.double()
    y = r * torch.rsqrt(r.pow(2).mean(-1, keepdim=True) + 1e-5) * w.double()
    torch.testing.assert_close(got.double(), y, rtol=2 ** -8, atol=2 ** -16)


def off_by(t, n):
    """``t`` from ``n`` elements behind an aligned address on."""
    flat = torch.empty(t.numel() + n, dtype=t.dtype, device=DEV)
    flat[n:] = t.flatten()
    return flat[n:].view(t.shape)


def test_skinny_forms_take_any_alignment():
    x, w = (t.contiguous() for t in operands(64, 512))
    x = x[:5].contiguous()
    want = ops.rows_linear(x[:, :256].contiguous(), w[:, :256].contiguous())
    a = off_by(x[:, :256], 4)
    b = off_by(w[:, :256], 4)
    assert not ops.rows_fit(a, b)
    for got in (ops.skinny_linear(a, b), ops.skinny2_linear(a, b),
                ops.linear_auto(a, b)):
        assert torch.equal(got, want)
    gu = torch.cat([x[:, :256], x[:, 256:]], 1)
    assert torch.equal(
        ops.skinny2_silu_linear(gu, b),
        ops.skinny2_silu_linear(gu, w[:, :256].contiguous()))


@pytest.mark.parametrize("M,N,K,fits", [
    # as timed beside the library
    (1, 4096, 14336, True), (64, 28672, 4096, True), (1, 256, 8192, True),
    (64, 256, 8192, False), (1, 64, 14336, False), (64, 512, 14336, True),
    (16, 20480, 3072, True), (64, 20480, 3072, False),
    (1, 20480, 8192, False), (64, 24576, 1024, True),
    (64, 10240, 256, False), (64, 10240, 4096, True),
    (128, 4096, 4096, True), (128, 16384, 2048, True),
    (128, 8192, 2048, False), (128, 12288, 4096, False),
    (128, 20480, 4096, False), (128, 57344, 5120, False),
    (128, 128256, 4096, True), (65, 2048, 2048, False)])
def test_rows_that_fit_are_the_faster_ones(M, N, K, fits):
    assert ops._rows_faster(M, N, K) == fits
    x = torch.empty(M, K, dtype=torch.bfloat16, device=DEV)
    assert ops.rows_fit(x, torch.empty(N, K, dtype=torch.bfloat16,
                                       device=DEV)) == fits


def test_weights_elsewhere_are_refused():
    x, w = operands(64, 128)
    with pytest.raises(RuntimeError):
        ops.rows_linear(x, w.cpu())


# tiles of 48 and 64 rows by 16 to 64 rows of w: their edges, a last one with few
# rows, one panel, fewer steps of K than waves, odd numbers of them
TALL = [(65, 4, 64), (65, 2048, 192), (96, 2044, 320), (97, 2052, 64),
        (128, 3076, 448), (129, 2048, 2048), (191, 2048, 128),
        (192, 3072, 1088), (193, 3072, 256), (256, 4096, 320),
        (257, 2040, 704), (96, 6160, 576), (128, 8192, 192), (768, 1024, 512),
        (767, 260, 3136), (129, 2048, 6144)]


@pytest.mark.parametrize("M,N,K", TALL)
def test_rows_tall(M, N, K):
    gen = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=gen).to(torch.bfloat16).to(DEV)
    w = torch.randn(N, K, generator=gen).to(torch.bfloat16).to(DEV)
    want = x.double() @ w.double().T
    got = torch.ops.rlli.rows_tall(x, w, False)
    close(got, want, K ** 0.5)
    # of the 16-bit product, in f32 and rounded once more
    relu2 = torch.ops.rlli.rows_tall(x, w, True)
    assert torch.equal(relu2, got.float().clamp(min=0).square()
                       .to(torch.bfloat16))


@pytest.mark.parametrize("N", [16, 264, 1040, 2048, 2056, 4100, 6160, 8192])
def test_every_tall_tile_is_in_one_round(N):
    work = torch.ops.rlli.rows_tall_work
    had = [work(M, N) for M in range(65, 800)]
    # from some number of rows on there is none, and until there more rows are
    # as much work or more
    some = [v for v in had if v]
    assert had == some + [0] * (len(had) - len(some))
    assert all(64 <= v <= 128 for v in some)


@pytest.mark.parametrize("M,N,K,fits", [
    (65, 2048, 1024, True), (768, 1024, 1024, True), (769, 256, 1024, False),
    (64, 2048, 2048, False), (320, 2048, 2048, True), (512, 2048, 2048, False),
    (320, 3072, 2048, False), (256, 4096, 2048, True), (96, 256, 2048, False),
    (128, 8192, 2048, True), (129, 8192, 2048, False), (80, 2048, 3072, False),
    (65, 3072, 3072, True), (128, 6144, 4096, True), (65, 8192, 4096, False),
    (129, 6144, 4096, False), (128, 1536, 4096, False), (65, 2048, 4160, True),
    (384, 2048, 6144, True), (385, 2048, 6144, False), (65, 2048, 6208, False),
    (128, 2112, 5120, False), (65, 2048, 2080, False)])
def test_tall_where_it_is_the_faster_one(M, N, K, fits):
    assert ops._tall_faster(M, N, K) == fits


def test_tall_refuses():
    x, w = operands(64, 128)
    for a, b in [(x, w.cpu()), (x.float(), w.float()), (x[:, :64], w[:, :64]),
                 (x, w[:62]), (x[:0], w), (x.repeat(60, 1), w.repeat(60, 1)),
                 (off_by(x, 4), w)]:
        with pytest.raises(RuntimeError):
            torch.ops.rlli.rows_tall(a, b, False)
