"""Steps of gated linear attention by workgroups of 1024 and of 256 threads:
states around the line between them, columns that do not divide the threads."""

import pytest
import torch

import resilient_llm_amd.ops as ops
from nesizen_util import BF16, F32
from test_mix_ops import gla_case, rel, tol


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("dim,vdim,rank", [
    (128, 256, 8), (127, 256, 24), (164, 200, 40), (256, 256, 64),
    (252, 130, 33)])
def test_steps(dim, vdim, rank, dtype):
    T, H = 9, 2
    *inputs, eps, want, S = gla_case(T, H, dim, vdim, rank, 8.0, 1.0,
                                     dim + rank, dtype)
    proj, a2, b, norm = (t.cuda() for t in inputs)
    st = torch.full((3, H, dim, -(-vdim // 4) * 4), float("nan"),
                    device="cuda")
    slot = torch.tensor([1], dtype=torch.int32, device="cuda")
    got = torch.cat([
        ops.gla_decode(proj[p:p + 1].contiguous(), a2, b, norm, st, slot,
                       torch.tensor([p], dtype=torch.int32, device="cuda"),
                       vdim, 8.0, eps) for p in range(T)])
    # the bounds of the longer runs over the same steps
    assert rel(got, want) < tol(dtype)
    assert rel(st[1, :, :, :vdim], S) < 1e-5
