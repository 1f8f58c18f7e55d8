"""The library's product with its choice kept by shape: what F.linear gives,
whatever the operands, streams and threads; tiles where that choice would sum
parts in a workspace."""

import threading

import pytest
import torch
import torch.nn.functional as F

from resilient_llm_amd import ops

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
    wrong = []

    def run(n):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            got = [(m, ops.library_linear(x[:m], w))
                   for m in range(1 + n, 1200, 2)]
            s.synchronize()
        # (a row's sum may be in another order with another number of rows)
        wrong.extend(m for m, y in got if not torch.allclose(
            y.float(), want[:m].float(), rtol=2 ** -7, atol=2 ** -14))
    threads = [threading.Thread(target=run, args=(i % 2,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
