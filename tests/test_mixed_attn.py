"""Attention of prompt rows and decoding sequences in one launch, against each by
itself: any division of either, sequences that end where units and waves do."""

import pytest
import torch

from resilient_llm_amd import ops
from resilient_llm_amd.ops import ref

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BS = 16


def step(n_q, n_kv, D, lens, portions, fp8, room=0):
    """A step's qkv, cache, tiles and tables on the CPU; ``portions``: (tokens
    before it, rows) of each prompt."""
    gen = torch.Generator().manual_seed(len(lens) + D)
    seen = lens + [s + n for s, n in portions]
    width = max(max(-(-n // BS) for n in seen), room)
    pages = len(seen) * width
    k, v = (torch.randn(pages, n_kv, BS, D, generator=gen)
            .to(torch.float8_e4m3fn if fp8 else torch.bfloat16)
            for _ in "kv")
    tables = torch.randperm(pages, generator=gen).to(torch.int32) \
        .view(len(seen), width)
    B, tiles, row = len(lens), [], len(lens)
    for b, (start, n) in enumerate(portions):
        for at in range(0, n, 32):
            tiles.append((row + at, start + at, min(32, n - at), b))
        row += n
    qkv = torch.randn(row, (n_q + 2 * n_kv) * D, generator=gen) \
        .to(torch.bfloat16)
    return (qkv, k, v, *torch.tensor(tiles, dtype=torch.int32).T.contiguous(),
            tables[B:].contiguous(), tables[:B].contiguous(),
            torch.tensor(lens, dtype=torch.int32), B, D ** -0.5, n_q)


def on_gpu(args):
    return [a.to(DEV) if isinstance(a, torch.Tensor) else a for a in args]


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("n_q,n_kv,D", [(32, 8, 128), (8, 1, 64), (8, 2, 128),
                                        (16, 2, 64)])
@pytest.mark.parametrize("lens,portions", [
    ([1], [(400, 1)]),
    ([31, 32, 33, 256, 257, 1100], [(383, 33), (0, 64), (900, 31)]),
    ([40] * 70 + [700], [(500, 40)])], ids=str)
def test_both(n_q, n_kv, D, lens, portions, fp8):
    args = step(n_q, n_kv, D, lens, portions, fp8)
    qkv, k, v, row0, pos0, nrows, btrow, pre, dec, dec_lens, B, scale, _ = args
    want = ref.prefill_paged_attn(qkv, k, v, row0, pos0, nrows, btrow, pre,
                                  scale, n_q)
    want[:B] = ref.decode_attn(qkv[:B, :n_q * D].reshape(B, n_q, D), k, v, dec,
                               dec_lens, scale).reshape(B, -1)
    gpu = on_gpu(args)
    ops.load_extension(required=True)
    # the rule's division, whole sequences and tiles, and many parts of either
    for plan in ([], [1, 0], [1, 3], [3, 64]):
        got = torch.ops.rlli.mixed_attn_qkv(*gpu, plan)
        # weights and outputs are each rounded to bf16 (2^-9 of them), values
        # are of size one and weights sum to one
        torch.testing.assert_close(got.cpu().float(), want.float(),
                                   atol=2 ** -7, rtol=2 ** -7)


def test_what_goes_apart():
    """Sizes that the launch does not take: the two ops, with their results."""
    ops.load_extension(required=True)
    for n_q, n_kv, portions in ((8, 4, [(400, 40)]), (8, 2, [(0, 40)]),
                                (32, 8, [(0, 2000)])):
        gpu = on_gpu(step(n_q, n_kv, 64, [100, 30], portions, False))
        with pytest.raises(RuntimeError, match="division"):
            torch.ops.rlli.mixed_attn_qkv(*gpu, [1, 0])
        want = ops.prefill_paged_attn(*gpu[:8], *gpu[-2:])
        ops.decode_attn_qkv_out(gpu[0][:2], *gpu[1:3], *gpu[8:10], *gpu[-2:],
                                want)
        assert torch.equal(ops.mixed_attn_qkv(*gpu), want)


@pytest.mark.parametrize("n_q,n_kv,D,lens,portions,apart", [
    # many short sequences, tiles that have more parts alone; and not
    (64, 8, 128, [16] * 200, [(0, 512)], True),
    (8, 1, 128, [16] * 4, [(0, 2048)], True),
    (32, 8, 128, [1500, 900, 1100], [(1500, 300)], False),
    (32, 8, 64, [300] * 30, [(600, 64)], False)])
def test_which_sizes_go_apart(n_q, n_kv, D, lens, portions, apart):
    gpu = on_gpu(step(n_q, n_kv, D, lens, portions, n_kv == 1))
    # (a step's tables of either kind have the pages of their longest)
    gpu[8] = gpu[8][:, :-(-max(lens) // BS)].contiguous()
    ops.load_extension(required=True)
    torch.ops.rlli.mixed_attn_qkv(*gpu, [1, 0])      # sizes that it takes
    torch.cuda.synchronize()
    with torch.profiler.profile() as prof:
        ops.mixed_attn_qkv(*gpu)
        torch.cuda.synchronize()
    names = [e.key for e in prof.key_averages()]
    assert any("mixed_attn_kernel" in n for n in names) != apart
    assert any("prefill_flash_kernel" in n for n in names) == apart


def test_no_tokens():
    """Sequences without tokens come out as zero, cut or whole."""
    args = on_gpu(step(8, 2, 64, [0, 300, 0], [(400, 5)], False, room=40))
    ops.load_extension(required=True)
    for plan in ([], [1, 0], [2, 16]):
        got = torch.ops.rlli.mixed_attn_qkv(*args, plan)
        assert not got[[0, 2]].any() and got[1].any()


def test_operands_are_checked():
    args = on_gpu(step(8, 2, 64, [100, 30], [(400, 5)], False))
    for i, bad in ((9, args[9].long()), (8, args[8][:1]), (10, 99)):
        wrong = list(args)
        wrong[i] = bad
        with pytest.raises(RuntimeError):
            ops.mixed_attn_qkv(*wrong)
