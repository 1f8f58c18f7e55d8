"""Short prompts' layers launched at once: the same bits as op by op, weights
that the kernels for few rows do not take included."""

import dataclasses

import pytest
import torch

from resilient_llm_amd.engine import LLMEngine, PagedKVCache
from resilient_llm_amd.engine.batch import Portion, PromptRows
from resilient_llm_amd.models import LlamaForCausalLM, get_config

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def feed(model, prompts, at_once, kv_dtype):
    kv = PagedKVCache.for_model(model.config, 40, device=DEV,
                                kv_dtype=kv_dtype)
    kv.k.zero_()
    kv.v.zero_()
    engine = LLMEngine(model, kv, max_batch_size=32)
    model._prompt_rows, kept = at_once, model._prompt_rows
    try:
        logits = engine.feed([(str(i), p, [len(p) - 1])
                              for i, p in enumerate(prompts)])
    finally:
        model._prompt_rows = kept
    return [logits] + [t.view(torch.uint8) for t in (kv.k, kv.v)]


@pytest.mark.parametrize("kv_dtype", [torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("name", ["tiny", "tiny-128"])
@pytest.mark.parametrize("lens", [[1], [33], [20, 1, 43]], ids=str)
@pytest.mark.parametrize("shifted", [None, "qkv", "o", "gate_up", "down"])
def test_same_bits(name, lens, shifted, kv_dtype):
    model = LlamaForCausalLM(get_config(name), device=DEV,
                             dtype=torch.bfloat16, seed=1)
    assert model._prompt_rows(sum(lens))
    if shifted:
        w = model.params[f"l1.{shifted}"]
        buf = torch.empty(w.numel() + 1, dtype=w.dtype, device=DEV)
        model.params[f"l1.{shifted}"] = buf[1:].view(w.shape).copy_(w)
    prompts = [[(7 * i + n) % 500 + 5 for i in range(n)] for n in lens]
    one, apart = (feed(model, prompts, lambda rows: x, kv_dtype)
                  for x in (True, False))
    for a, b in zip(one, apart):
        assert torch.equal(a, b)


@pytest.mark.parametrize("name", ["tiny", "tiny-128"])
@pytest.mark.parametrize("heads", [(4, 4), (4, 2), (8, 1)], ids=str)
@pytest.mark.parametrize("lens", [[64], [32, 32], [31, 33], [2] * 32],
                         ids=lambda lens: f"{len(lens)}x{lens[0]}")
def test_rotation_inside(name, heads, lens):
    """Tiles of rows that end where keys' do, heads in groups of any size."""
    config = dataclasses.replace(get_config(name), n_heads=heads[0],
                                 n_kv_heads=heads[1])
    model = LlamaForCausalLM(config, device=DEV, dtype=torch.bfloat16, seed=1)
    assert model._prompt_rows(64)
    prompts = [[(7 * i + n) % 500 + 5 for i in range(n)] for n in lens]
    one, apart = (feed(model, prompts, lambda rows: x, torch.bfloat16)
                  for x in (True, False))
    for a, b in zip(one, apart):
        assert torch.equal(a, b)


def test_which_prompts():
    model = LlamaForCausalLM(get_config("tiny"), device=DEV,
                             dtype=torch.bfloat16)
    assert model._prompt_rows(64) and not model._prompt_rows(65)
    assert not model._prompt_rows(0)
    model.params["l1.o"].requires_grad_()
    assert not model._prompt_rows(8)


def test_one_token():
    """Of one row the norm is inside gate and up, in layers at once as well.
    Sums of squares in another order turn the rounding of one normed element in
    2^18 or so: 2000 rows of 4096."""
    config = dataclasses.replace(get_config("llama-3-8b"), n_layers=3,
                                 vocab_size=1005)
    model = LlamaForCausalLM(config, device=DEV, dtype=torch.bfloat16, seed=1)
    assert model._prompt_rows(1)
    w = model.params["l1.gate_up"]
    assert torch.ops.rlli.rows_norm_ok(*w.shape, True)
    kv = PagedKVCache.for_model(config, 4, device=DEV)
    ids = torch.arange(1005, dtype=torch.int32, device=DEV)
    first, rows = ids[:1], ids[:2]

    def logits(at_once):
        model._prompt_rows = lambda rows: at_once
        return torch.cat([model.forward_prefill(ids[i:i + 1], first, kv, first,
                                                rows)
                          for i in range(5, 1005)])
    assert torch.equal(logits(True), logits(False))


@pytest.mark.parametrize("n", [1, 64, 65, 700])
def test_tables_behind_a_busy_stream(n):
    """Tables are sent by copies that nobody waits for: made one after another
    while the stream is busy, each has its own values."""
    def tables(device, i):
        rows = PromptRows([Portion(0, i, n, 0, 1), Portion(n, 0, i + 1, 1, i)],
                          device)
        return [rows.tiles(64), rows.seqs(64), rows.spans(32), rows.pos0(),
                *rows.gathered(32)[:2], rows.vectors(16, 3)]
    x = torch.randn(4096, 4096, device="cuda")
    for _ in range(20):
        x = torch.mm(x, x) * 1e-3
    got = [tables("cuda", i) for i in range(30)]
    for i, made in enumerate(got):
        for g, want in zip(made, tables("cpu", i)):
            assert g.dtype == want.dtype and torch.equal(g.cpu(), want)


def test_tables_on_another_stream():
    """A table that a busy stream has not come to yet is none for others."""
    portions = [Portion(0, i, 40 + i, 0, i) for i in range(9)]
    rows, x = PromptRows(portions, "cuda"), torch.randn(4096, 4096,
                                                        device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.Stream()):
        for _ in range(40):
            x = torch.mm(x, x) * 1e-3
        first = rows.tiles(16)
    want = PromptRows(portions, "cpu").tiles(16)
    assert torch.equal(rows.tiles(16).cpu(), want)
    torch.cuda.synchronize()
    assert torch.equal(first.cpu(), want)


def test_tables_in_a_capture():
    """Tables that are there before a capture are taken as they are in it."""
    rows = PromptRows([Portion(0, 0, 70, 0, 0)], "cuda")
    want = rows.tiles(16), rows.seqs(64), rows.pos0()
    graph, out = torch.cuda.CUDAGraph(), torch.zeros_like(want[0])
    with torch.cuda.graph(graph):
        got = rows.tiles(16), rows.seqs(64), rows.pos0()
        out.copy_(got[0])
    assert all(g is w for g, w in zip(got, want))
    for _ in range(3):
        out.zero_()
        graph.replay()
        assert torch.equal(out, want[0])
