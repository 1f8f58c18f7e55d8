"""The library's product with its choice kept by shape: what F.linear gives,
whatever the operands, streams and threads; tiles where that choice would sum
parts in a workspace."""

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

import pytest
import torch
import torch.nn.functional as F
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.autograd import forward_ad

from resilient_llm_amd import ops
from resilient_llm_amd.models import llama

DEV = "cuda:0"


def operands(M, N, K, dtype=torch.bfloat16, device=DEV):
    g = torch.Generator().manual_seed(M + N + K)
    return (torch.randn(M, K, generator=g).to(device, dtype),
            (torch.randn(N, K, generator=g) * K ** -0.5).to(device, dtype))


def close(got, x, w):
    # K f32 roundings of sums of size one, then half a step of bf16
    torch.testing.assert_close(got.double(), x.double() @ w.double().T,
                               rtol=2 ** -8, atol=2 ** -14)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (3, 7, 5), (65, 96, 72),
                                   (129, 6160, 2048), (777, 640, 1000)])
def test_as_linear(M, N, K):
    x, w = operands(M, N, K)
    for _ in range(2):
        assert torch.equal(ops.library_linear(x, w), F.linear(x, w))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1025, 4096, 14336), (4300, 4096, 14336),
                                   (4475, 1048, 8256), (3308, 6160, 2048)])
def test_many_rows(M, N, K):
    x, w = operands(M, N, K)
    close(ops.library_linear(x, w), x, w)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1700, 3072, 14336), (2600, 2560, 14336)])
def test_few_tiles_divide_k(M, N, K):
    """Whatever the library picks, tiles are not left to go through a long K where
    a few of them are all."""
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).bfloat16()
    w = (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16()
    got = ops.library_linear(x.to(DEV), w.to(DEV)).cpu()
    # (f32 here too: K roundings of sums of size one, then half a step of bf16)
    torch.testing.assert_close(got.float(), x.float() @ w.float().T,
                               rtol=2 ** -8, atol=2 ** -13)


@pytest.mark.parametrize("M,N,K,splits", [
    (1100, 64, 28672, 8), (1900, 1024, 28672, 6), (4300, 4096, 14336, 1),
    (6500, 5120, 2048, 1),
    # parts of more than 76 MiB are not made
    (2300, 4096, 28672, 1), (1025, 8192, 28672, 1), (2048, 2048, 28672, 4)])
def test_parts_of_tiles(M, N, K, splits):
    ops.load_extension(required=True)
    mh, nh, n = torch.ops.rlli.tiles_for_library(M, N, K)
    assert n == splits
    if splits > 1:
        tiles = -(-M // (64 * mh)) * -(-N // (128 * nh))
        assert tiles * n > 64


def test_other_operands_cpu():
    x, w = operands(5, 6, 7, torch.float32, "cpu")
    assert torch.equal(ops.library_linear(x, w), F.linear(x, w))


@pytest.mark.gpu
def test_other_operands():
    x, w = operands(66, 64, 128)
    for a, b in [(x[:0], w), (x[:, :64], w[:, :64]), (x[1:], w[2:]),
                 (x.flatten()[1:1 + 65 * 128].view(65, 128), w),
                 (x.view(2, 33, 128), w), (x.float(), w.float()),
                 (x.t().contiguous().t(), w)]:
        assert torch.equal(ops.library_linear(a, b), F.linear(a, b))
    x.requires_grad_()
    ops.library_linear(x, w).sum().backward()
    assert x.grad is not None
    with pytest.raises(RuntimeError):
        ops.library_linear(x.detach(), w[:, :64])


@pytest.mark.gpu
def test_streams_and_threads():
    """More shapes than are kept, from four threads on streams of their own."""
    w = operands(1, 64, 64)[1]
    x = operands(1200, 64, 64)[0]
    want = F.linear(x, w)
    torch.cuda.synchronize()

    def run(n):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            got = [(m, ops.library_linear(x[:m], w))
                   for m in range(1 + n, 1200, 2)]
            s.synchronize()
        # (a row's sum may be in another order with another number of rows)
        return len(got), [m for m, y in got if not torch.allclose(
            y.float(), want[:m].float(), rtol=2 ** -7, atol=2 ** -14)]
    with ThreadPoolExecutor(4) as pool:
        ran = list(pool.map(run, [0, 1, 0, 1]))
    assert ran == [(600, []), (599, [])] * 2


@pytest.mark.gpu
def test_plans_of_the_last_sizes():
    """Of more shapes than are kept, the least recently used go, and those one by
    one."""
    kept = torch.ops.rlli.library_plans_kept
    w = operands(1, 64, 64)[1]
    x = operands(1200, 64, 64)[0]
    for m in range(1, 1201):
        ops.library_linear(x[:m], w)
    assert kept() == 1024


# rows that rows_tall, the library and (N not a multiple of 128) tiles take
FORMS = [(200, 2048, 2048), (1000, 4096, 4096), (2048, 6160, 2048)]


@pytest.mark.parametrize("M,N,K", FORMS)
def test_sizes_of_a_trace(M, N, K):
    """Tensors without memory, as of a trace and of vmap, go F.linear's way."""
    with FakeTensorMode():
        x = torch.empty(M, K, dtype=torch.bfloat16, device=DEV)
        w = torch.empty(N, K, dtype=torch.bfloat16, device=DEV)
        assert llama._linear(x, w).shape == (M, N)
        many = torch.func.vmap(lambda a: llama._linear(a, w))(
            x.expand(3, M, K))
        assert many.shape == (3, M, N) and many.dtype == x.dtype


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(65, 256, 64), (130, 640, 1000),
                                   (600, 2064, 64)])
def test_tangents(M, N, K):
    x, w = operands(M, N, K)
    t = torch.randn_like(x)
    want = F.linear(t, w)
    with forward_ad.dual_level():
        y = llama._linear(forward_ad.make_dual(x, t), w)
        tangent = forward_ad.unpack_dual(y).tangent
    assert torch.equal(tangent, want)
    y, tangent = torch.func.jvp(lambda a: llama._linear(a, w), (x,), (t,))
    assert torch.equal(tangent, want)
    close(y, x, w)


@pytest.mark.gpu
def test_autocast():
    x, w = operands(130, 640, 1000)
    with torch.autocast("cuda", torch.float16):
        got, want = ops.library_linear(x, w), F.linear(x, w)
    assert got.dtype == want.dtype and torch.equal(got, want)


OWN_SPACE = """
import torch
from resilient_llm_amd import ops
ops.load_extension(required=True)
print(torch.ops.rlli.library_plans_on())
"""


@pytest.mark.parametrize("own", [None, "HIPBLASLT_WORKSPACE_SIZE",
                                 "CUBLASLT_WORKSPACE_SIZE"])
def test_workspace_of_the_process(own):
    """One that sets the library's workspace itself has no plans of ours."""
    env = {k: v for k, v in os.environ.items() if "WORKSPACE_SIZE" not in k}
    if own:
        env[own] = str(128 << 10)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    ran = subprocess.run([sys.executable, "-c", OWN_SPACE], cwd=root, env=env,
                         timeout=100, capture_output=True, text=True)
    assert ran.stdout.split() == [str(own is None)], ran.stderr[-2000:]
