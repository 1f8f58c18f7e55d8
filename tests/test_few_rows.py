"""A mixed step whose prompt rows are few takes the decode kernel: the rows
give what tiles of them give."""

import pytest
import torch

from resilient_llm_amd import ops
from resilient_llm_amd.engine import LLMEngine, PagedKVCache
from resilient_llm_amd.models import LlamaForCausalLM, get_config



def tables_of(device):
    """Two decoding sequences and tiles of 3, 0 and 2 rows; rows 5 and 8
    belong to none."""
    def i32(x):
        return torch.tensor(x, dtype=torch.int32, device=device)
    return ops.mixed_row_tables(
        9, 2, i32([[7, 8, 9]] * 3), i32([40, 0, 5]), i32([2, 0, 6]),
        i32([16, 3, 0]), i32([3, 0, 2]), i32([1, -9, 0]),
        i32([[1, 2], [3, 4]]))


def test_row_tables():
    tables, lens = tables_of("cpu")
    assert lens.tolist() == [40, 0, 17, 18, 19, 0, 1, 2, 0]
    assert tables.tolist() == [[7, 8, 9]] * 2 + [[3, 4, 0]] * 3 + [[0] * 3] \
        + [[1, 2, 0]] * 2 + [[0] * 3]


@pytest.mark.gpu
def test_row_tables_on_the_device():
    for got, want in zip(tables_of("cuda:0"), tables_of("cpu")):
        assert torch.equal(got.cpu(), want)


@pytest.mark.gpu
def test_rows_of_no_tile(monkeypatch):
    """Tiles that leave rows out, a decoding sequence without tokens: as
    tiles have it for the others."""
    cfg = get_config("tiny-128")
    model = LlamaForCausalLM(cfg, device="cuda:0", dtype=torch.bfloat16,
                             seed=1)

    def i32(*x):
        return torch.tensor(x, dtype=torch.int32, device="cuda:0")
    got = []
    for few in (True, False):
        monkeypatch.setattr(model, "_few_rows", lambda *a: few)
        kv = PagedKVCache.for_model(cfg, 8, device="cuda:0")
        kv.k.zero_()
        kv.v.zero_()
        got.append(model.forward_mixed(
            i32(*range(5, 12)), i32(3, 0, 0, 1, 2, 0, 1), kv,
            i32(19, 32, 48, 49, 50, 64, 65), 2, i32([1], [2]), i32(4, 0),
            i32(2, 5), i32(0, 0), i32(2, 2), i32(0, 1), i32([3], [4]),
            torch.tensor([2, 3, 5, 6], device="cuda:0")))
    torch.testing.assert_close(got[0], got[1], atol=0.05, rtol=0.05)


@pytest.mark.gpu
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
