"""A norm that two products share: the first's result into the streams, the
second's factor of a row, against both in 64 bits; rows and columns where tiles and
waves end."""

import pytest
import torch

from nesizen_util import EVEN, check, expected, for_dtype, make_engine, tokens_of
from resilient_llm_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF16 = torch.bfloat16


def operands(M, N, K, nxt, S):
    gen = torch.Generator().manual_seed(M + N + S)

    def rnd(*shape, std=1.0):
        return torch.randn(*shape, generator=gen) * std
    return (rnd(M, K).to(BF16), rnd(N, K, std=K ** -0.5).to(BF16),
            3 * rnd(M, S, N), rnd(S, S), rnd(S), rnd(S), 1 + 0.1 * rnd(N),
            rnd(nxt, N, std=N ** -0.5).to(BF16))


@pytest.mark.parametrize("M", [1, 15, 16, 17, 32])
@pytest.mark.parametrize("N,K,nxt,S", [
    (64, 64, 16, 1), (192, 128, 4100, 2), (2048, 3072, 6144, 3),
    (4096, 320, 68, 4)])
def test_shared_norm(M, N, K, nxt, S):
    x, w, streams, mix, out_w, in_w, gain, w2 = operands(M, N, K, nxt, S)
    dev = [t.to(DEV) for t in (x, w, streams, mix, out_w, in_w, gain)]
    assert ops.rows_streams_fit(dev[0], dev[1], dev[2], w2.to(DEV))
    y = x.double() @ w.double().T
    want = torch.einsum("st,msn->mtn", mix.double(), streams.double()) \
        + out_w.double()[:, None] * y[:, None]
    u = (in_w.double()[:, None] * want).sum(1)
    h, ss = ops.rows_linear_streams_(*dev)
    # 32-bit sums of K products of size one
    torch.testing.assert_close(dev[2].cpu().double(), want, atol=2e-5,
                               rtol=2e-5)
    torch.testing.assert_close(ss.cpu().double().sum(0)[:M],
                               u.pow(2).sum(1), atol=0, rtol=2e-5)
    torch.testing.assert_close(h.cpu().double(), u * gain.double(), atol=2e-5,
                               rtol=2 ** -8 + 2e-5)
    got = ops.rows_linear_scaled_relu2(h, ss, 1e-5, w2.to(DEV)).cpu().double()
    inv = torch.rsqrt(u.pow(2).mean(1, keepdim=True) + 1e-5)
    full = torch.relu((u * gain.double() * inv) @ w2.double().T)
    # h is rounded to bf16: a product is off by the sum of N random errors of up
    # to 2^-9 N^-1/2, of which five deviations are below 5 2^-9; its square, a bf16
    # number, is off by 2 a d + d^2 and 2^-9 of it, its root by d and 2^-10 of it
    torch.testing.assert_close(got.sqrt(), full, atol=5 * 2 ** -9,
                               rtol=2 ** -10)


def test_streams_and_gains_anywhere():
    """They may start at any float, as those of a step by itself."""
    args = [t.to(DEV) for t in operands(17, 256, 2048, 1024, 2)][:-1]
    off = list(args)
    for i in (2, 3, 4, 5, 6):
        off[i] = torch.empty(args[i].numel() + 1, device=DEV)[1:] \
            .view(args[i].shape).copy_(args[i])
    want, got = (ops.rows_linear_streams_(*a) for a in (args, off))
    # (sums of squares of rows that there are)
    assert torch.equal(got[0], want[0])
    assert torch.equal(got[1][:, :17], want[1][:, :17])
    assert torch.equal(off[2], args[2])


def test_what_does_not_fit():
    x, w, streams, mix, out_w, in_w, gain, w2 = (
        t.to(DEV) for t in operands(8, 256, 2048, 1024, 2))
    assert ops.rows_streams_fit(x, w, streams, w2)
    assert not ops.rows_streams_fit(x.repeat(5, 1), w, streams, w2)
    assert not ops.rows_streams_fit(x, w, streams, w2.float())
    assert not ops.rows_streams_fit(x, w, streams, w2[:, :128])
    assert not ops.rows_streams_fit(x, w, streams.repeat(1, 3, 1), w2)
    assert not ops.rows_streams_fit(x.float(), w, streams, w2)
    for i, bad in ((2, streams.half()), (3, mix[:1]), (6, gain[:-1]),
                   (2, streams[:4]), (0, x.cpu())):
        args = [x, w, streams, mix, out_w, in_w, gain]
        args[i] = bad
        with pytest.raises(RuntimeError):
            ops.rows_linear_streams_(*args)
    h, ss = ops.rows_linear_streams_(x, w, streams, mix, out_w, in_w, gain)
    for bad in (ss[:-1], ss.double(), ss[:, :8]):
        with pytest.raises(RuntimeError):
            ops.rows_linear_scaled_relu2(h, bad, 1e-5, w2)


def test_model_takes_it(monkeypatch):
    """Of 32 rows the layers with a dense feed-forward share its norm, of 33 none."""
    config = for_dtype(EVEN, BF16)
    dense = sum(x["mlp"] is not None for x in config["layers"])
    engine, w = make_engine(config, DEV, BF16)
    rows, fused = [], ops.rows_linear_streams_

    def counted(x, *rest):
        rows.append(x.shape[0])
        return fused(x, *rest)
    monkeypatch.setattr(ops, "rows_linear_streams_", counted)
    for n, calls in ((1, dense), (32, dense), (33, 0)):
        rows.clear()
        t = tokens_of(config, n, n)
        got = engine.feed([(f"{n}", t, range(n))], [f"{n}"])
        assert rows == [n] * calls
        check(got, expected(config, w, t), BF16, f"{n} rows")
