"""A decoded row's attention and the product behind it: parts put together
inside the product, whole sequences, weights that it does not take."""

import pytest
import torch

from resilient_llm_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def setup(n, width, n_q, n_kv, D, N, fp8):
    gen = torch.Generator().manual_seed(n)
    blocks = width // 16
    k, v = (torch.randn(blocks, n_kv, 16, D, generator=gen)
            .to(torch.float8_e4m3fn if fp8 else torch.bfloat16).to(DEV)
            for _ in "kv")
    table = torch.randperm(blocks, generator=gen).to(torch.int32)[None]
    at = max(n - 1, 0)
    slot = table[0, at // 16] * 16 + at % 16
    cs = ops.build_cos_sin(width, D, 10000.0).to(DEV)
    qkv = torch.randn(3, 1, (n_q + 2 * n_kv) * D, generator=gen).to(DEV)
    w = (torch.randn(N, n_q * D, generator=gen) * (n_q * D) ** -0.5).to(
        torch.bfloat16).to(DEV)

    def one(x):
        return torch.tensor([x], dtype=torch.int32, device=DEV)
    return (qkv, one(at), cs, k, v, slot[None].to(torch.int32).to(DEV),
            table.contiguous().to(DEV), one(n), D ** -0.5, n_q), w


# one part; two to sixty-four of them, across batches of eight; no tokens
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("n", [0, 1, 250, 257, 1000, 2049, 2305, 8190])
@pytest.mark.parametrize("n_q,n_kv,D,N", [
    (32, 8, 128, 4096), (8, 1, 64, 48), (16, 16, 128, 512), (4, 1, 128, 64)])
def test_parts_in_the_product(n, n_q, n_kv, D, N, fp8):
    args, w = setup(n, 8192, n_q, n_kv, D, N, fp8)
    caches = [t.clone() for t in args[3:5]]
    out = ops.decode_attn_rope_qkv(*args)
    kept = [t.clone() for t in args[3:5]]
    for t, c in zip(args[3:5], caches):
        t.copy_(c)
    got = ops.decode_attn_rope_linear(*args, w)
    for t, c in zip(args[3:5], kept):
        assert torch.equal(t.view(torch.uint8), c.view(torch.uint8))
    got = got.sum(0) if got.dim() == 3 else got
    # Parts in another order of sums turn the rounding of one output in 2^8 or
    # so: sqrt(2^-8) 2^-8 of the result, which its few largest elements exceed
    # fourfold, and the product's f32 sums.
    want = out.double() @ w.double().T
    torch.testing.assert_close(got.double(), want, rtol=0,
                               atol=2 ** -10 * float(out.abs().max()) + 1e-9)


def test_other_weights():
    args, w = setup(1000, 2048, 8, 2, 128, 64, False)
    want = ops.decode_attn_rope_qkv(*args).double() @ w.double().T
    buf = torch.empty(w.numel() + 1, dtype=w.dtype, device=DEV)
    for other in (buf[1:].view(w.shape).copy_(w), w.T.contiguous().T):
        got = ops.decode_attn_rope_linear(*args, other)
        torch.testing.assert_close(got.double(), want, rtol=2 ** -7,
                                   atol=2 ** -8)


def test_several_rows_go_apart():
    args, w = setup(1000, 2048, 8, 2, 128, 64, False)
    two = [torch.cat([t, t], 1 if t.dim() == 3 else 0) if i in (0, 1, 5, 6, 7)
           else t for i, t in enumerate(args)]
    # the second row's key goes where neither looks
    two[5][1] = args[6][0, 100] * 16
    want = ops.decode_attn_rope_qkv(*two).double() @ w.double().T
    got = ops.decode_attn_rope_linear(*two, w)
    torch.testing.assert_close(got.sum(0).double(), want, rtol=0, atol=2 ** -10)
