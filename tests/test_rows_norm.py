"""The norm inside the product of one row that follows it: the ends of a
thread's pieces, parts in one and in several batches."""

import pytest
import torch

from resilient_llm_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def inputs(n, N, K):
    gen = torch.Generator().manual_seed(n)

    def draw(*shape):
        return torch.randn(*shape, generator=gen)
    parts = draw(n, 1, K).to(DEV)
    residual = draw(1, K).to(torch.bfloat16).to(DEV)
    gain = (1 + 0.1 * draw(K)).to(torch.bfloat16).to(DEV)
    w = (draw(N, K) * K ** -0.5).to(torch.bfloat16).to(DEV)
    return parts, residual, gain, w


@pytest.mark.parametrize("n,N,K,silu", [
    (4, 64, 128, False), (1, 60, 192, False), (8, 3072, 2048, False),
    (9, 4100, 2112, False), (4, 6144, 4096, False), (5, 512, 4160, False),
    (2, 3072, 8192, False), (4, 25632, 4096, True), (17, 10304, 2112, True),
    (8, 25616, 320, True), (8, 16384, 2048, True)])
def test_rows_norm_linear(n, N, K, silu):
    parts, residual, gain, w = inputs(n, N, K)
    assert ops.rows_norm_fit(parts, residual, w, silu)
    kept = residual.clone()
    got, after = ops.rows_norm_linear(parts, residual, gain, 1e-5, w, silu)
    assert torch.equal(residual, kept)
    whole = residual.clone()
    h = ops.rmsnorm_residual_(parts, whole, gain, 1e-5)
    # the same sums, in the same order
    assert torch.equal(after, whole)
    want = h.double() @ w.double().T
    if silu:
        g, u = want.chunk(2, 1)
        want = torch.nn.functional.silu(g) * u
    else:
        got = got.sum(0)
    # The sum of squares in another order may turn the rounding of one element
    # of h in 2^8 or so: sqrt(2^-8) 2^-8 of the result, of size one, which its
    # few largest elements exceed fourfold.  Of silu, its own rounding.
    torch.testing.assert_close(got.double(), want, atol=2 ** -10,
                               rtol=2 ** -8 if silu else 0)


@pytest.mark.parametrize("N,K,silu", [
    (20480, 4096, False), (4096, 64, False), (57344, 4096, True),
    (1024, 2048, True), (4096, 8256, False)])
def test_which_products(N, K, silu):
    assert not torch.ops.rlli.rows_norm_ok(N, K, silu)
    residual = torch.zeros(1, K, dtype=torch.bfloat16, device=DEV)
    w = torch.zeros(N, K, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(RuntimeError, match="rows_norm_ok"):
        ops.rows_norm_linear(torch.zeros(2, 1, K, device=DEV), residual,
                             w[0].clone(), 1e-5, w, silu)


def test_operands_are_checked():
    parts, residual, gain, w = inputs(4, 64, 128)
    two = residual.expand(2, -1).contiguous()
    for bad in ((parts[:, :, :64], residual, gain), (parts.double(), residual,
                gain), (parts, residual, gain[:64]), (parts[0], residual,
                gain), (parts, residual, gain.cpu()), (parts, two, gain)):
        with pytest.raises(RuntimeError):
            ops.rows_norm_linear(*bad, 1e-5, w, False)


def test_gain_of_any_alignment():
    parts, residual, gain, w = inputs(4, 64, 128)
    odd = torch.cat([gain[:1], gain])[1:]
    assert odd.data_ptr() % 16
    for got, want in zip(
            ops.rows_norm_linear(parts, residual, odd, 1e-5, w, False),
            ops.rows_norm_linear(parts, residual, gain, 1e-5, w, False)):
        assert torch.equal(got, want)
