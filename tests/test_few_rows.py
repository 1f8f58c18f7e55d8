"""A mixed step whose prompt rows are few takes the decode kernel: the rows
give what tiles of them give."""

import pytest
import torch

from resilient_llm_amd.engine import LLMEngine, PagedKVCache
from resilient_llm_amd.models import LlamaForCausalLM, get_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("portions", [[5], [1, 16, 3], [4, 4, 4, 4, 4]],
                         ids=str)
def test_few_rows(portions, monkeypatch):
    cfg = get_config("tiny-128")
    model = LlamaForCausalLM(cfg, device="cuda:0", dtype=torch.bfloat16,
                             seed=1)
    gen = torch.Generator().manual_seed(0)

    def tokens(n):
        return torch.randint(5, 500, (n,), generator=gen).tolist()
    heads = [tokens(20 + 50 * i) for i in range(len(portions))]
    tails = [tokens(n) for n in portions]
    decoded = tokens(33)
    got = []
    for few in (True, False):
        if not few:
            monkeypatch.setattr(model, "_few_rows", lambda *a: False)
        e = LLMEngine(model, PagedKVCache.for_model(
            cfg, 128, device="cuda:0"), max_batch_size=8)
        e.feed([(f"p{i}", h, []) for i, h in enumerate(heads)]
               + [("d", decoded, [])])
        assert not few or model._few_rows(sum(portions), len(portions))
        # (a decoding row goes first)
        got.append(e.feed(
            [("d", [7], [0])] + [(f"p{i}", t, list(range(len(t))))
                                 for i, t in enumerate(tails)]))
    # two layers of 16-bit activations; tiles round queries and weights
    torch.testing.assert_close(got[0], got[1], atol=0.05, rtol=0.05)
