"""Tiled expert products where the order of the tiles matters: experts whose
last tile is just under, at and just over half full, without rows, with one
row, and with more tiles than a group of four."""

import pytest
import torch

import nesizen_plain as plain
import resilient_llm_amd.ops as ops
from nesizen_util import BF16
from test_mix_ops import D64, pack, rel, rnd

COUNTS = [
    # tiles of 128 rows
    [64, 65, 0, 1, 128, 129, 640, 63],
    [192, 193, 191, 127, 0, 0, 1300, 192],
    # of 256 rows
    [128, 129, 127, 0, 1, 256, 257, 2600],
    [384, 385, 383, 640, 0, 1281, 900, 255],
    [256, 257, 300, 290, 512, 1, 255, 529],
]


@pytest.mark.gpu
# (from 2048 on, up to 300 rows an expert, blocks of w start K at their own steps)
@pytest.mark.parametrize("W,ff", [(320, 192), (64, 1152), (2112, 192),
                                  (64, 2112)])
@pytest.mark.parametrize("counts", COUNTS, ids=str)
def test_tiles_of_all_fills(counts, W, ff):
    E, limit = len(counts), 0.8
    g = torch.Generator().manual_seed(sum(counts))
    owner = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    owner = owner[torch.randperm(len(owner), generator=g)]
    T = len(owner)
    h = rnd((T, W), 1, BF16)
    h[:, :E] = 0
    h[torch.arange(T), owner] = 2.0
    router = torch.zeros(E, W, dtype=BF16)
    router[torch.arange(E), torch.arange(E)] = 2.0
    gate, up = (rnd((E, ff, W), s, BF16, 1.5 * W ** -0.5) for s in (2, 3))
    down = rnd((E, W, ff), 4, BF16, ff ** -0.5)
    w_up, w_down = pack(gate, up, down)
    got = ops.moe_experts(h.cuda(), router.cuda(), w_up.cuda(), w_down.cuda(),
                          1, limit).cpu()[:, 0]
    s = torch.sigmoid(torch.tensor(4.0, dtype=D64))
    for e in range(E):
        t = torch.nonzero(owner == e)[:, 0]
        if len(t):
            want = plain.clamped_expert(
                s.expand(len(t), 1) * h[t].double(), gate[e].double(),
                up[e].double(), down[e].double(), limit)
            # the bound of the other bf16 expert tests: the hidden values and
            # the result are rounded once each
            assert rel(got[t], want) < 8e-3, e
