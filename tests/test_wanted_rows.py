"""Logits of some rows of a step against those of all its rows: the last layer
is for the wanted rows alone where they are few (models/mixed.py narrow_to)."""

import pytest
import torch

from resilient_llm_amd.engine import LLMEngine, PagedKVCache
from resilient_llm_amd.models import build_model, get_config
from resilient_llm_amd.models.mixed import narrow_to

TARGETS = [pytest.param("cpu", torch.float32, id="cpu-f32"),
           pytest.param("cuda:0", torch.bfloat16, id="cuda-bf16",
                        marks=pytest.mark.gpu)]


def fed(model, device, dtype, portions, want):
    """Logits of feeding each request's tokens at once."""
    config = model.config
    kv = PagedKVCache.for_model(config, 64, device=device, state_slots=8)
    if dtype == torch.float32 and hasattr(kv, "k"):
        kv.k, kv.v = kv.k.float(), kv.v.float()
    e = LLMEngine(model, kv, max_batch_size=4, enable_prefix_caching=False)
    return e.feed([(f"r{i}", t, w) for i, (t, w) in
                   enumerate(zip(portions, want))]).float().cpu()


@pytest.mark.parametrize("device,dtype", TARGETS)
@pytest.mark.parametrize("name", ["tiny", "tiny-128", "nesizen-tiny"])
@pytest.mark.parametrize("lens,want", [
    ([65], [[64]]), ([64], [[63]]), ([130, 1, 40], [[129, 0], [0], [39]]),
    ([33, 33], [list(range(0, 32)), [32]]), ([90], [[3, 3, 89]]),
    ([40, 40], [[], [39]])])
def test_some_rows_as_of_all(name, lens, want, device, dtype):
    model = build_model(get_config(name), device=device, dtype=dtype, seed=3)
    g = torch.Generator().manual_seed(sum(lens))
    V = model.config.vocab_size
    toks = [torch.randint(5, V, (n,), generator=g).tolist() for n in lens]
    all_rows = fed(model, device, dtype, toks, [range(n) for n in lens])
    starts = [sum(lens[:i]) for i in range(len(lens))]
    ref = all_rows[[s + r for s, w in zip(starts, want) for r in w]]
    got = fed(model, device, dtype, toks, want)
    # the same products with their sums in another order: of K terms in f32
    # up to K 2^-24, K 1024; of 16 bits half a unit in the last place of each
    # of a few roundings in the last layer
    rel = float((got - ref).norm() / ref.norm())
    assert rel < (1e-4 if dtype == torch.float32 else 0.02), rel


def test_which_rows():
    rows = torch.arange(32)
    assert narrow_to(rows, 65) and narrow_to(rows[:1], 4096)
    assert not narrow_to(rows, 64) and not narrow_to(None, 4096)
    assert not narrow_to(rows[:0], 4096) and not narrow_to(torch.arange(33), 65)


def test_other_indices():
    """What the last norm's rows may be chosen by beside a list of them, they are
    chosen by there."""
    assert not narrow_to(torch.tensor(3), 4096)
    assert not narrow_to(torch.zeros(2, 3, dtype=torch.long), 4096)
    assert not narrow_to(torch.zeros(128, dtype=torch.bool), 4096)
    assert not narrow_to(slice(0, 3), 4096) and not narrow_to([3, 5], 4096)
