"""What the host makes of a step's portions: positions, slots and tiles of every
token, and their way to the device."""

import pytest
import torch

from resilient_llm_amd.engine import LLMEngine, PagedKVCache
from resilient_llm_amd.engine.batch import _numbers, sent
from resilient_llm_amd.models import build_model, get_config




@pytest.mark.parametrize("name", ["tiny", "nesizen-tiny"])
@pytest.mark.parametrize("parts", [[[1]], [[16], [15]], [[17, 1, 30]],
                                   [[5, 40], [64], [33, 2]]])
def test_rows_of_a_step(name, parts):
    """Portions of several requests, each behind what it has cached."""
    model = build_model(get_config(name), dtype=torch.float32, seed=1)
    kv = PagedKVCache.for_model(model.config, 64, device="cpu", state_slots=8)
    if hasattr(kv, "k"):
        kv.k, kv.v = kv.k.float(), kv.v.float()
    e = LLMEngine(model, kv, enable_prefix_caching=False)
    calls = []
    for f in ("forward_prefill", "forward_mixed", "forward_decode"):
        real = getattr(model, f, None)
        if real is not None:
            def call(*a, real=real, f=f, **kw):
                calls.append((f, a))
                return real(*a, **kw)
            setattr(model, f, call)
    at = [0] * len(parts)
    for step in range(max(len(p) for p in parts)):
        now = [(i, p[step]) for i, p in enumerate(parts) if step < len(p)]
        calls.clear()
        e.feed([(f"r{i}", list(range(5, 5 + n)), [n - 1]) for i, n in now])
        (f, a), = calls
        pos, slots = a[1].tolist(), a[3].tolist()
        # rows of single tokens behind a prefix come first
        order = ([(i, n) for i, n in now if n == 1 and at[i]]
                 + [(i, n) for i, n in now if n > 1 or not at[i]])
        want = [(i, at[i] + k) for i, n in order for k in range(n)]
        assert pos == [p for _, p in want]
        blocks = {i: e._fed[f"r{i}"].blocks for i, _ in now}
        assert slots == [blocks[i][p // 16] * 16 + p % 16 for i, p in want]
        if f == "forward_mixed" and name == "tiny":
            nd, row0, pos0, nrows, btrow = a[4], *(t.tolist() for t in a[7:11])
            tiles = [(b, r, p, min(32, n - o)) for b, (i, n, r) in enumerate(
                     (i, n, sum(m for _, m in order[:k]))
                     for k, (i, n) in enumerate(order) if k >= nd)
                     for o in range(0, n, 32)
                     for r, p in [(r + o, at[i] + o)]]
            assert list(zip(btrow, row0, pos0, nrows)) == tiles
        for i, n in now:
            at[i] += n


@pytest.mark.parametrize("device", ["cpu", pytest.param(
    "cuda:0", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("dtype", [torch.int32, torch.long, torch.float32])
@pytest.mark.parametrize("n", [0, 1, 512, 513, 2000])
def test_sent(n, dtype, device):
    values = [(-1) ** i * i * 1000 for i in range(n)]
    got = sent(values, dtype, device)
    assert got.dtype == dtype and got.device == torch.device(device)
    assert got.tolist() == values
    pairs = list(zip(values, values[::-1]))
    if pairs:
        assert sent(pairs, dtype, device).tolist() == [list(p) for p in pairs]


@pytest.mark.parametrize("device", ["cpu", pytest.param(
    "cuda:0", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("dtype", [torch.int32, torch.long])
def test_sent_with_a_fraction(dtype, device):
    values = [1] * 600 + [2.7, -3.5]
    got = sent(values, dtype, device)
    assert got.dtype == dtype and got.tolist() == [1] * 600 + [2, -3]


def test_long_lists_of_whole_numbers():
    values = list(range(-300, 300))
    for dtype in (torch.int32, torch.long):
        assert _numbers(values, dtype).tolist() == values
        assert _numbers(values[:512], dtype) is None
        assert _numbers(values + [0.5], dtype) is None
    assert _numbers(values, torch.float32) is None
