"""A captured decode step's state: batches that fill their bucket or leave rows
of it, tables as wide as the buffers or narrower, more of either than a
workgroup has threads; against the same by tensor ops on the CPU."""

import pytest
import torch

from resilient_llm_amd import ops

GOLDEN = 0x9E3779B97F4A7C15 - (1 << 64)


def state(gen, rows, width):
    def ints(*shape, dtype=torch.int32):
        return torch.randint(0, 4000, shape, generator=gen, dtype=dtype)
    return (ints(rows), ints(rows), ints(rows, width),
            torch.rand(rows, generator=gen), ints(rows, dtype=torch.int64),
            ints(rows))


SIZES = [(1, 1, 1, 1, 1), (1, 1, 1, 7, 8), (4, 2, 3, 64, 64),
         (64, 37, 40, 255, 256), (256, 256, 256, 257, 600),
         (65, 64, 65, 512, 513), (8, 0, 1, 5, 9)]


def check_load(dev, rows, batch, bucket, wide, width, slots, change=None):
    gen = torch.Generator().manual_seed(rows + wide)
    to, new = state(gen, rows, width), state(gen, batch, wide)
    if not slots:
        new = (*new[:5], None)
    want = [t.clone() for t in to]
    for t, n in zip(want, new):
        if n is None:
            continue
        if n.dim() == 2:
            t[:batch, :wide] = n
            t[:batch, wide:] = 11
        else:
            t[:batch] = n
    for t, fill in zip(want, (0, 0, 11, 0, 0, 13)):
        t[batch:bucket] = fill
    got = [t.to(dev) for t in to]
    new = [n if n is None else n.to(dev) for n in new]
    if change:
        new = change(new)
    ops.decode_load(got, new, bucket, 11, 13)
    for g, w in zip(got, want):
        assert torch.equal(g.cpu(), w)


def check_step(dev, rows, width, block):
    gen = torch.Generator().manual_seed(rows)
    ids, pos, tables, _, seeds, tokens = state(gen, rows, width)
    # up to beyond the table's end, as padded rows get to
    pos = pos % (block * (width + 1))
    seeds = seeds * (1 << 50)
    block_of = (pos // block).clamp(max=width - 1).long()
    slots = tables[torch.arange(rows), block_of] * block + pos % block
    got = [t.clone().to(dev) for t in (ids, pos, tables, seeds, tokens)]
    s, n = ops.decode_begin(got[1], got[2], block)
    assert s.dtype == n.dtype == torch.int32
    assert torch.equal(s.cpu(), slots) and torch.equal(n.cpu(), pos + 1)
    ops.decode_advance_(got[0], got[1], got[3], got[4], GOLDEN)
    assert torch.equal(got[0].cpu(), tokens)
    assert torch.equal(got[1].cpu(), pos + 1)
    assert torch.equal(got[3].cpu(), seeds + GOLDEN)


@pytest.mark.parametrize("sizes", SIZES)
@pytest.mark.parametrize("slots", [False, True])
def test_load_cpu(sizes, slots):
    check_load("cpu", *sizes, slots)


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", SIZES)
@pytest.mark.parametrize("slots", [False, True])
def test_load(sizes, slots):
    check_load("cuda:0", *sizes, slots)


@pytest.mark.gpu
@pytest.mark.parametrize("change", [
    lambda new: [n if n is None else n.cpu() for n in new],
    lambda new: [new[0].long(), *new[1:]],
    lambda new: [*new[:2], new[2].T.contiguous().T, *new[3:]]])
def test_load_of_other_tensors(change):
    check_load("cuda:0", 8, 5, 8, 6, 9, True, change)


@pytest.mark.parametrize("rows,width,block", [(1, 1, 16), (65, 7, 16)])
def test_step_cpu(rows, width, block):
    check_step("cpu", rows, width, block)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,width,block", [
    (1, 1, 16), (1, 8, 16), (64, 512, 16), (65, 7, 8), (256, 33, 48)])
def test_step(rows, width, block):
    check_step("cuda:0", rows, width, block)
