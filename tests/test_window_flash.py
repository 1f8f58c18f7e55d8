"""Windowed prompt attention by transposed 32 x 32 scores: windows that end
within, at and behind tiles of keys, kept tokens in and behind the first
tile, rows that see nothing of a walked tile, every head grouping."""

import pytest
import torch

from nesizen_util import BF16
from test_mix_ops import Attn, rel, tol

# H, G, dim
HEADS = [(1, 1, 128), (4, 2, 64), (8, 2, 128), (8, 1, 64)]
# window, kept first tokens
MASKS = [(1, 0), (1, 4), (5, 70), (33, 0), (64, 1), (65, 64), (100, 65),
         (4000, 0)]


@pytest.mark.gpu
@pytest.mark.parametrize("sink", [False, True])
@pytest.mark.parametrize("H,G,dim", HEADS)
@pytest.mark.parametrize("window,keep", MASKS)
def test_masks_and_pieces(H, G, dim, window, keep, sink):
    T = 331
    a = Attn(T, H, G, dim, dim, 32, window, keep, "cuda", BF16, seed=dim + H)
    if sink:
        a.sink[0] = 30.0               # far above every score
    want = a.want(sink)
    p, got = 0, []
    for n in (1, 63, 66, 130, T - 260):
        got.append(a.run(p, n, sink=sink))
        p += n
    got = torch.cat(got).cpu()
    # one bound for each head, so that a sink that takes all cannot hide
    for h in range(H):
        cols = slice(h * dim, (h + 1) * dim)
        assert rel(got[:, cols], want[:, cols]) < tol(BF16), h
