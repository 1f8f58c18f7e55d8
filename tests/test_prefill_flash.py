"""Causal prompt attention at the sizes where its tiles end: 32 rows, 64
keys, sequences counted 64 at a time, pages of any size, every head group."""

import pytest
import torch

from resilient_llm_amd import ops
from resilient_llm_amd.ops import ref

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def close(got, want):
    # weights and outputs are each rounded to bf16 (2^-9 of them), values
    # are of size one and weights sum to one
    torch.testing.assert_close(got.cpu().float(), want.float(), atol=2 ** -7,
                               rtol=2 ** -7)


@pytest.mark.parametrize("n_q,n_kv,D", [
    (4, 1, 128), (8, 8, 64), (4, 2, 128), (8, 1, 64), (32, 8, 128)])
@pytest.mark.parametrize("lens", [
    [1], [31, 32, 33], [63, 64, 65], [0, 5, 0, 129], [3] * 66 + [40]],
    ids=str)
def test_batch_rows(n_q, n_kv, D, lens):
    gen = torch.Generator().manual_seed(len(lens))
    T = sum(lens)
    qkv = torch.randn(T, (n_q + 2 * n_kv) * D, generator=gen) \
        .to(torch.bfloat16)
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
    # scores far apart: maxima move from tile to tile
    for scale in (D ** -0.5, -1.5):
        got = ops.prefill_attn_qkv(qkv.to(DEV), cu.to(DEV), scale, n_q, n_kv,
                                   D)
        q, k, v = (t.reshape(T, -1, D) for t in torch.split(
            qkv, [n_q * D, n_kv * D, n_kv * D], 1))
        close(got, ref.prefill_attn(q, k, v, cu, scale).reshape(T, -1))


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("n_q,n_kv,D,bs", [
    (8, 2, 128, 16), (8, 1, 64, 16), (2, 1, 128, 8), (3, 3, 64, 4),
    (4, 1, 128, 32)])
def test_pages(n_q, n_kv, D, bs, fp8):
    gen = torch.Generator().manual_seed(D + bs)
    # (position of the first row, rows) of each sequence
    seqs = [(0, 33), (63, 1), (64, 32), (97, 31)]
    width = max(-(-(s + n) // bs) for s, n in seqs)
    pages = len(seqs) * width
    k, v = (torch.randn(pages, n_kv, bs, D, generator=gen) for _ in "kv")
    k, v = (t.to(torch.float8_e4m3fn if fp8 else torch.bfloat16)
            for t in (k, v))
    tables = torch.randperm(pages, generator=gen).to(torch.int32) \
        .view(len(seqs), width)
    T = sum(n for _, n in seqs)
    qkv = torch.randn(T, (n_q + 2 * n_kv) * D, generator=gen) \
        .to(torch.bfloat16)
    tiles, row = [], 0
    for b, (start, n) in enumerate(seqs):
        tiles += [(row + o, start + o, min(32, n - o), b)
                  for o in range(0, n, 32)]
        row += n
    t = torch.tensor(tiles, dtype=torch.int32).t().contiguous()
    got = ops.prefill_paged_attn(
        qkv.to(DEV), k.to(DEV), v.to(DEV), *t.to(DEV), tables.to(DEV),
        D ** -0.5, n_q)
    k, v = (x.float().to(torch.bfloat16) for x in (k, v))
    close(got, ref.prefill_paged_attn(qkv, k, v, *t, tables, D ** -0.5, n_q))


@pytest.mark.parametrize("n_q,n_kv,D", [(4, 1, 128), (8, 1, 64)])
@pytest.mark.parametrize("lens", [[385], [448, 449], [384, 1, 800]], ids=str)
def test_two_waves_per_head(n_q, n_kv, D, lens):
    """Few workgroups: tiles of keys go to two waves in turn; odd and even
    counts of tiles, rows that the second wave has nothing for."""
    test_batch_rows(n_q, n_kv, D, lens)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("D,bs", [(128, 16), (64, 16), (128, 8)])
def test_two_waves_per_head_over_pages(D, bs, fp8):
    n_q, n_kv = 8, 2
    gen = torch.Generator().manual_seed(bs)
    seqs = [(0, 33), (63, 1), (447, 66), (512, 31), (0, 400)]
    width = -(-544 // bs)
    k, v = (torch.randn(len(seqs) * width, n_kv, bs, D, generator=gen)
            .to(torch.float8_e4m3fn if fp8 else torch.bfloat16) for _ in "kv")
    tables = torch.randperm(len(seqs) * width, generator=gen) \
        .to(torch.int32).view(len(seqs), width)
    qkv = torch.randn(sum(n for _, n in seqs), (n_q + 2 * n_kv) * D,
                      generator=gen).to(torch.bfloat16)
    tiles, row = [], 0
    for b, (start, n) in enumerate(seqs):
        tiles += [(row + o, start + o, min(32, n - o), b)
                  for o in range(0, n, 32)]
        row += n
    t = torch.tensor(tiles, dtype=torch.int32).t().contiguous()
    got = ops.prefill_paged_attn(
        qkv.to(DEV), k.to(DEV), v.to(DEV), *t.to(DEV), tables.to(DEV),
        D ** -0.5, n_q)
    k, v = (x.float().to(torch.bfloat16) for x in (k, v))
    close(got, ref.prefill_paged_attn(qkv, k, v, *t, tables, D ** -0.5, n_q))


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("n_q,n_kv,D,bs", [(4, 1, 128, 16), (8, 2, 64, 16),
                                           (8, 1, 128, 8)])
@pytest.mark.parametrize("seqs", [
    [(2000, 40)], [(2047, 1)], [(0, 65), (1023, 2), (255, 31), (8100, 33)]],
    ids=str)
def test_keys_in_parts(n_q, n_kv, D, bs, fp8, seqs):
    """Workgroups that share a tile's keys: up to sixteen parts, sequences too
    short for them, rows that see nothing of a part's last keys."""
    gen = torch.Generator().manual_seed(bs)
    width = -(-max(s + n for s, n in seqs) // bs)
    k, v = (torch.randn(len(seqs) * width, n_kv, bs, D, generator=gen)
            .to(torch.float8_e4m3fn if fp8 else torch.bfloat16) for _ in "kv")
    tables = torch.randperm(len(seqs) * width, generator=gen) \
        .to(torch.int32).view(len(seqs), width)
    # a row in front and one behind that are nobody's
    T = sum(n for _, n in seqs) + 2
    qkv = torch.randn(T, (n_q + 2 * n_kv) * D, generator=gen) \
        .to(torch.bfloat16)
    tiles, row = [], 1
    for b, (start, n) in enumerate(seqs):
        tiles += [(row + o, start + o, min(32, n - o), b)
                  for o in range(0, n, 32)]
        row += n
    t = torch.tensor(tiles, dtype=torch.int32).t().contiguous()
    got = ops.prefill_paged_attn(
        qkv.to(DEV), k.to(DEV), v.to(DEV), *t.to(DEV), tables.to(DEV),
        D ** -0.5, n_q)
    k, v = (x.float().to(torch.bfloat16) for x in (k, v))
    want = ref.prefill_paged_attn(qkv, k, v, *t, tables, D ** -0.5, n_q)
    close(got[1:-1], want[1:-1])


def test_row_offsets_of_any_device_and_count():
    gen = torch.Generator().manual_seed(1)
    qkv = torch.randn(45, 6 * 64, generator=gen).to(torch.bfloat16).to(DEV)
    cu = torch.tensor([0, 13, 45], dtype=torch.int32)
    args = 0.125, 4, 1, 64
    assert torch.equal(ops.prefill_attn_qkv(qkv, cu, *args),
                       ops.prefill_attn_qkv(qkv, cu.to(DEV), *args))
    for none in (cu[:1], cu[:0]):
        for t in (none, none.to(DEV)):
            with pytest.raises(RuntimeError, match="without a sequence"):
                ops.prefill_attn_qkv(qkv, t, *args)
            assert ops.prefill_attn_qkv(qkv[:0], t, *args).shape == (0, 256)


def off_by(t, n):
    """``t`` from ``n`` elements behind an aligned address on."""
    flat = torch.empty(t.numel() + n, dtype=t.dtype, device=DEV)
    flat[n:] = t.to(DEV).flatten()
    return flat[n:].view(t.shape)


def test_operands_of_any_alignment():
    gen = torch.Generator().manual_seed(2)
    qkv = torch.randn(45, 6 * 64, generator=gen).to(torch.bfloat16)
    cu = torch.tensor([0, 13, 45], dtype=torch.int32).to(DEV)
    args = 0.125, 4, 1, 64
    want = ops.prefill_attn_qkv(qkv.to(DEV), cu, *args)
    assert torch.equal(ops.prefill_attn_qkv(off_by(qkv, 4), cu, *args), want)
    k, v = (torch.randn(4, 1, 16, 64, generator=gen).to(torch.bfloat16)
            for _ in "kv")
    tiles = torch.tensor([[0, 0, 32, 0], [32, 32, 13, 0]],
                         dtype=torch.int32).t().contiguous().to(DEV)
    table = torch.tensor([[2, 0, 3, 1]], dtype=torch.int32).to(DEV)

    def paged(k, v):
        return ops.prefill_paged_attn(qkv.to(DEV), k, v, *tiles, table, 0.125,
                                      4)
    assert torch.equal(paged(off_by(k, 4), off_by(v, 4)),
                       paged(k.to(DEV), v.to(DEV)))
