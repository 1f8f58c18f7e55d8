"""Decode attention where its units, parts and pages end: 32 tokens, 256
tokens, lengths counted 64 sequences at a time, pages of any size; queries
as rows and as the parts of a product."""

import pytest
import torch

from resilient_llm_amd import ops
from resilient_llm_amd.ops import ref

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

LENS = {
    "whole": [1, 31, 32, 33, 64, 255, 256],
    "parts": [257, 1, 1000, 33, 4097, 0, 512],
    "many": [0, 0] + [40] * 66 + [700, 1],
}


def setup(lens, n_q, n_kv, D, bs, fp8, width=None):
    gen = torch.Generator().manual_seed(D + bs + len(lens))
    need = [-(-n // bs) for n in lens]
    pages = sum(need) + 1
    k, v = (torch.randn(pages, n_kv, bs, D, generator=gen) for _ in "kv")
    dtype = torch.float8_e4m3fn if fp8 else torch.bfloat16
    order = torch.randperm(pages, generator=gen).to(torch.int32)
    tables = torch.zeros(len(lens), width or max(need), dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        tables[i, :n] = order[at:at + n]
        at += n
    qkv = torch.randn(len(lens), (n_q + 2 * n_kv) * D, generator=gen)
    return (k.to(dtype), v.to(dtype), tables, torch.tensor(
        lens, dtype=torch.int32), qkv.to(torch.bfloat16))


def exact(q, k, v, tables, lens, scale):
    """In 64 bits; sequences without tokens give zeros."""
    out = torch.zeros(q.shape, dtype=torch.float64)
    for b, n in enumerate(lens.tolist()):
        if n:
            keys, values = (
                t[tables[b].long()].transpose(0, 1)
                .reshape(t.shape[1], -1, t.shape[3])[:, :n].float().double()
                .repeat_interleave(q.shape[1] // t.shape[1], 0)
                for t in (k, v))
            w = torch.softmax(torch.einsum("hd,hnd->hn", q[b].double(), keys)
                              * scale, -1)
            out[b] = torch.einsum("hn,hnd->hd", w, values)
    return out


def close(got, want):
    # f32 throughout, rounded to bf16 once
    torch.testing.assert_close(got.cpu().double(), want, rtol=2 ** -8,
                               atol=2 ** -14)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("lens", LENS)
@pytest.mark.parametrize("n_q,n_kv,D,bs", [
    (8, 2, 128, 16), (8, 1, 64, 16), (2, 2, 128, 16), (2, 1, 64, 8),
    (4, 1, 128, 32)])
def test_cached(n_q, n_kv, D, bs, lens, fp8):
    k, v, tables, n, qkv = setup(LENS[lens], n_q, n_kv, D, bs, fp8)
    q = qkv[:, :n_q * D].reshape(-1, n_q, D).contiguous()
    # scores far apart as well
    for scale in (D ** -0.5, 1.0):
        got = ops.decode_attn(q.to(DEV), k.to(DEV), v.to(DEV),
                              tables.to(DEV), n.to(DEV), scale)
        close(got, exact(q, k, v, tables, n, scale))


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("lens", ["whole", "parts"])
@pytest.mark.parametrize("n_q,n_kv,D,bs", [
    (8, 2, 128, 16), (8, 1, 64, 16), (4, 1, 128, 8)])
def test_fused(n_q, n_kv, D, bs, lens, fp8):
    """Rotation, append and the new token; its slot held NaN."""
    lens = [max(1, x) for x in LENS[lens]]
    k, v, tables, n, qkv = setup(lens, n_q, n_kv, D, bs, fp8)
    pos = n - 1
    slots = tables.gather(1, (pos // bs).long()[:, None])[:, 0] * bs + pos % bs
    cs = ref.build_cos_sin(max(lens), D)
    args = [x.to(DEV) for x in (pos, cs)]
    tail = [x.to(DEV) for x in (slots, tables, n)]

    def run(rows):
        kc, vc = k.clone(), v.clone()
        for t in (kc, vc):
            t.float()
            raw = t.view(torch.uint8 if fp8 else torch.int16)
            raw[(slots // bs).long(), :, (slots % bs).long()] = \
                0x7f if fp8 else 0x7fc0
        kc, vc = kc.to(DEV), vc.to(DEV)
        out = ops.decode_attn_rope_qkv(rows, *args, kc, vc, *tail,
                                       D ** -0.5, n_q)
        return out, kc, vc
    got, kc, vc = run(qkv.to(DEV))
    kr, vr = k.clone(), v.clone()
    q, key, value = (t.reshape(len(lens), -1, D) for t in torch.split(
        qkv, [n_q * D, n_kv * D, n_kv * D], 1))
    rot = ref._rotate(torch.cat([q, key], 1).float(), pos, cs)
    at = (slots // bs).long(), slice(None), (slots % bs).long()
    kr[at] = rot[:, n_q:].to(k.dtype)
    vr[at] = value.to(v.dtype)
    # a rotation's rounding may fall either way
    torch.testing.assert_close(kc.cpu().float(), kr.float(), rtol=2 ** -3
                               if fp8 else 2 ** -7, atol=2 ** -9)
    assert torch.equal(vc.cpu().float(), vr.float())
    close(got.view(-1, n_q, D), exact(rot[:, :n_q], kc.cpu(), vr, tables, n,
                                      D ** -0.5))
    # the same rows as a sum
    rows = qkv.float().to(DEV)
    part = torch.randn(rows.shape, device=DEV).to(torch.bfloat16).float() / 8
    again, k2, v2 = run(torch.stack([rows - part, part]))
    assert torch.equal(again, got)
    assert torch.equal(k2.float(), kc.float())
    assert torch.equal(v2.float(), vc.float())


def test_rows_of_one_sequence():
    """Rows appended first and attended like decoded tokens: the same bits,
    whichever way they came, as no sequence of this batch is cut into other
    parts than in a smaller one."""
    lens = [37, 38, 39, 300, 301]
    k, v, tables, n, qkv = (t.to(DEV) for t in setup(
        lens, 8, 2, 128, 16, False))
    tables[1:3] = tables[0:1].clone()         # three tokens of one sequence
    tables[4] = tables[3]
    pos = n - 1
    slots = tables.gather(1, (pos // 16).long()[:, None])[:, 0] * 16 \
        + pos % 16
    cs = ref.build_cos_sin(512, 128, device=DEV)
    kc, vc = k.clone(), v.clone()
    got = ops.decode_attn_rows_qkv(qkv.clone(), pos, cs, kc, vc, slots,
                                   tables, n, 0.1, 8)
    for order in ([0, 3], [1, 4], [2]):
        at = torch.tensor(order, device=DEV)
        want = ops.decode_attn_rope_qkv(
            qkv[at], pos[at], cs, k, v, slots[at], tables[at], n[at], 0.1, 8)
        assert torch.equal(got[at], want)
    assert torch.equal(k, kc) and torch.equal(v, vc)


@pytest.mark.parametrize("D", [64, 128])
def test_8_bit_codes_come_out_as_they_are(D):
    codes = torch.arange(256).to(torch.uint8).view(torch.float8_e4m3fn)
    # (the two NaNs as zeros)
    codes = torch.where(codes.float().isnan(), torch.zeros(256),
                        codes.float()).to(torch.float8_e4m3fn)
    rows = codes.view(256 // D, 1, 1, D)
    k = torch.zeros(256 // D, 1, 16, D).to(torch.float8_e4m3fn)
    v = k.clone()
    k[:, :, :1], v[:, :, :1] = rows, rows
    n = torch.ones(256 // D, dtype=torch.int32)
    q = torch.ones(256 // D, 2, D, dtype=torch.bfloat16)
    got = ops.decode_attn(q.to(DEV), k.to(DEV), v.to(DEV),
                          torch.arange(256 // D, dtype=torch.int32)[:, None]
                          .contiguous().to(DEV), n.to(DEV), 0.01)
    want = rows.float().view(-1, 1, D).expand(-1, 2, -1)
    assert torch.equal(got.cpu().float(), want)


def fused_args(lens, n_q=8, n_kv=2, D=128):
    k, v, tables, n, qkv = (t.to(DEV) for t in setup(lens, n_q, n_kv, D, 16,
                                                     False))
    pos = n - 1
    slots = tables.gather(1, (pos // 16).long()[:, None])[:, 0] * 16 \
        + pos % 16
    return qkv, pos, ref.build_cos_sin(max(lens), D, device=DEV), k, v, \
        slots, tables, n


def test_buffers_longer_than_the_batch():
    qkv, pos, cs, k, v, slots, tables, n = fused_args([37, 300, 5, 64])
    want = ops.decode_attn_rope_qkv(qkv[:3], pos[:3], cs, k.clone(), v.clone(),
                                    slots[:3], tables[:3], n[:3], 0.1, 8)
    got = ops.decode_attn_rope_qkv(qkv[:3], pos, cs, k.clone(), v.clone(),
                                   slots, tables, n, 0.1, 8)
    assert torch.equal(got, want)
    want = ops.decode_attn_qkv(qkv[:3], k, v, tables[:3], n[:3], 0.1, 8)
    assert torch.equal(ops.decode_attn_qkv(qkv[:3], k, v, tables, n, 0.1, 8),
                       want)
    # a values' cache of more pages
    more = torch.cat([v, v[:1]])
    assert torch.equal(ops.decode_attn_qkv(qkv[:3], k, more, tables, n, 0.1,
                                           8), want)


@pytest.mark.parametrize("short", range(4))
def test_buffers_shorter_than_the_batch(short):
    qkv, pos, cs, k, v, slots, tables, n = fused_args([37, 300, 5])
    bufs = [pos, slots, tables, n]
    bufs[short] = bufs[short][:2]
    pos, slots, tables, n = bufs
    with pytest.raises(RuntimeError):
        ops.decode_attn_rope_qkv(qkv, pos, cs, k, v, slots, tables, n, 0.1, 8)


def test_rows_of_other_ranks_are_refused():
    qkv, pos, cs, k, v, slots, tables, n = fused_args([37, 300, 5])
    # one row per sequence in between, no parts, f32 that is not parts
    for rows, n_pos in ((qkv[:, None], 1), (qkv.float()[None][:0], 3),
                        (qkv.float(), 3)):
        with pytest.raises(RuntimeError):
            ops.decode_attn_rope_qkv(rows, pos[:n_pos], cs, k, v,
                                     slots[:n_pos], tables, n, 0.1, 8)
    with pytest.raises(RuntimeError):
        ops.decode_attn_qkv(qkv[:, None], k, v, tables, n, 0.1, 8)
    res = torch.zeros(3, 64, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(RuntimeError):
        ops.rmsnorm_residual_(torch.zeros(0, 3, 64, device=DEV), res,
                              res[0].clone())


@pytest.mark.parametrize("n_q,n_kv,D,L", [
    (32, 8, 128, 1000), (32, 4, 128, 70), (32, 4, 64, 1000), (16, 8, 64, 40),
    (8, 8, 128, 300)])
def test_queries_and_weights_keep_32_bits(n_q, n_kv, D, L):
    """Of outputs with a relative error e, 2 e / 2^-8 are not the bf16 number
    nearest to the exact one: 2^-12 for f32 sums with e = 2^-21, 2^-8 if
    queries and weights had 16 bits."""
    k, v, tables, n, qkv = setup([L] * 32, n_q, n_kv, D, 16, False)
    q = qkv[:, :n_q * D].reshape(32, n_q, D)
    cs = ref.build_cos_sin(L, D)
    slots = tables[:, (L - 1) // 16] * 16 + (L - 1) % 16
    kc, vc = k.to(DEV), v.to(DEV)
    got = ops.decode_attn_rope_qkv(
        qkv.to(DEV), (n - 1).to(DEV), cs.to(DEV), kc, vc, slots.to(DEV),
        tables.to(DEV), n.to(DEV), D ** -0.5, n_q)
    c, s = cs[L - 1].double().chunk(2)
    a, b = q.double().chunk(2, -1)
    want = exact(torch.cat([a * c - b * s, b * c + a * s], -1), kc.cpu(),
                 vc.cpu(), tables, n, D ** -0.5)
    off = got.cpu().view_as(q) != want.to(torch.bfloat16)
    assert off.double().mean() < 2 ** -10


@pytest.mark.parametrize("n_q,n_kv,D,L", [(8, 2, 128, 70), (8, 1, 64, 600),
                                          (2, 2, 64, 40)])
def test_infinite_keys_and_values(n_q, n_kv, D, L):
    """A key that is -inf where queries are positive takes no weight; values
    that are infinite make their channel so.  Queries have 8 bits here, so
    that all parts but the first are zero."""
    k, v, tables, n, qkv = setup([L] * 3, n_q, n_kv, D, 16, False)
    q = qkv[:, :n_q * D].reshape(3, n_q, D).contiguous()
    q[..., 5] = q[..., 5].abs() + 0.5
    page, at = tables[:, 1].long(), 3
    k[page, :, at, 5] = -torch.inf
    v[page, :, at + 1, 7] = torch.inf
    v[page, :, at + 2, 9] = -torch.inf
    got = ops.decode_attn(q.to(DEV), k.to(DEV), v.to(DEV), tables.to(DEV),
                          n.to(DEV), D ** -0.5)
    want = exact(q, k, v, tables, n, D ** -0.5)
    assert want[..., 7].isinf().all() and want[..., :5].isfinite().all()
    close(got, want)


@pytest.mark.parametrize("n_q,n_kv,D,bs", [(8, 2, 128, 16), (8, 1, 64, 16),
                                           (2, 2, 64, 8)])
def test_newest_value_infinite(n_q, n_kv, D, bs):
    """An infinite value makes its channel so also as the newest token's, wherever
    in a unit of 32 tokens that is."""
    k, v, tables, n, qkv = setup([1, 31, 32, 33, 70, 257, 1000], n_q, n_kv, D,
                                 bs, False)
    new = qkv[:, (n_q + n_kv) * D:].view(len(n), n_kv, D)
    new[..., 7], new[..., 9] = torch.inf, -torch.inf
    pos = n - 1
    slots = tables.gather(1, (pos // bs).long()[:, None])[:, 0] * bs + pos % bs
    cs = ref.build_cos_sin(1000, D)
    kc, vc = k.to(DEV), v.to(DEV)
    got = ops.decode_attn_rope_qkv(
        qkv.to(DEV), pos.to(DEV), cs.to(DEV), kc, vc, slots.to(DEV),
        tables.to(DEV), n.to(DEV), D ** -0.5, n_q).view(-1, n_q, D)
    q = qkv[:, :n_q * D].reshape(-1, n_q, D)
    want = exact(ref._rotate(q.float(), pos, cs), kc.cpu(), vc.cpu(), tables, n,
                 D ** -0.5)
    assert (want[..., 7] == torch.inf).all() and want[..., :7].isfinite().all()
    close(got, want)
    # and where the cache has it
    got = ops.decode_attn(q.to(DEV), kc, vc, tables.to(DEV), n.to(DEV),
                          D ** -0.5)
    close(got, exact(q, kc.cpu(), vc.cpu(), tables, n, D ** -0.5))


def test_parts_follow_from_the_batch():
    """Together the sequences have parts of ten units, alone of eight: the
    sums' order differs, and with it the last bit of some outputs."""
    lens = [4097, 4000, 4097, 4096, 3000, 700]
    qkv, pos, cs, k, v, slots, tables, n = fused_args(lens, 8, 8, 64)
    got = ops.decode_attn_rope_qkv(qkv, pos, cs, k.clone(), v.clone(), slots,
                                   tables, n, 0.1, 8)
    for b in range(len(lens)):
        at = slice(b, b + 1)
        want = ops.decode_attn_rope_qkv(
            qkv[at], pos[at], cs, k.clone(), v.clone(), slots[at], tables[at],
            n[at], 0.1, 8)
        # each rounded to bf16 once, of sums that agree to about 2^-20
        torch.testing.assert_close(got[at].float(), want.float(),
                                   rtol=2 ** -7, atol=2 ** -14)
