"""The residual streams' step over f32 parts of a product, against the same
step over their sum: widths of every launch shape, odd counts of parts, a
subset of rows."""

import subprocess
import sys

import pytest
import torch

import resilient_llm_amd.ops as ops
from nesizen_util import F32
from test_mix_ops import rel, rnd


def test_the_op_is_there_on_first_use():
    """In a process of its own: the library may be loaded here already."""
    code = (
        "import torch, resilient_llm_amd.ops as ops\n"
        "d = 'cuda:0' if torch.cuda.is_available() else 'cpu'\n"
        "x, y = torch.ones(3, 2, 8, device=d), torch.ones(4, 3, 8, device=d)\n"
        "one = torch.ones(8, device=d)\n"
        "h = ops.hyper_step(x, y, one[:4].view(2, 2).clone(), one[:2].clone(),"
        " None, one, 0.0, split=True)\n"
        "assert h.dtype == torch.bfloat16 and bool((h == 1).all()), h\n"
        "assert bool((x == 6).all()), x\n")
    subprocess.run([sys.executable, "-c", code], check=True, timeout=300)


@pytest.mark.gpu
@pytest.mark.parametrize("S,W,n", [(1, 40, 1), (2, 264, 3), (3, 1032, 6),
                                   (2, 2048, 8), (5, 4096, 2), (8, 4104, 5)])
def test_step_over_parts(S, W, n):
    T, eps = 5, 3e-4
    x, y = rnd((T, S, W), 1, F32), rnd((n, T, W), 2, F32)
    mix, outw, inw = (rnd(s, 3, F32) for s in ((S, S), (S,), (S,)))
    gain = 1 + rnd((W,), 4, F32, 0.3)
    rows = torch.tensor([4, 1])
    want_x = x.double()
    args = (mix.double(), outw.double())
    total = y.double().sum(0)
    new = torch.einsum("st,nsw->ntw", args[0], want_x) \
        + args[1][None, :, None] * total[:, None]

    def normed(u):
        return u / (u.pow(2).mean(-1, keepdim=True) + eps).sqrt() \
            * gain.double()

    dev = [t.cuda() for t in (x, y, mix, outw, inw, gain)]
    last = ops.hyper_step(*dev[:4], None, dev[5], eps, rows.cuda(),
                          keep=False, split=True)
    assert last.dtype == torch.bfloat16
    # one rounding to bf16 of at most 2^-9 of each value
    assert rel(last, normed(new.sum(1))[rows]) < 2 ** -9
    assert torch.equal(dev[0].cpu(), x)                    # left alone
    h = ops.hyper_step(*dev, eps, split=True)
    assert rel(h, normed(torch.einsum("s,tsw->tw", inw.double(), new))) \
        < 2 ** -9
    assert rel(dev[0], new) < 3e-6
    with pytest.raises(RuntimeError):
        ops.hyper_step(dev[0], dev[1][:, :4].contiguous(), *dev[2:], eps,
                       split=True)
