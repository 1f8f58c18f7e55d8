"""Each mixed-layer mechanism alone, CPU form and HIP kernels, against the
plain equations: streams, windowed attention, gated linear attention,
experts, sampler.  Inputs are made so that one wrong key, edge, sink,
decay or route shows."""

import math

import pytest
import torch

import nesizen_plain as plain
import resilient_llm_amd.ops as ops
from nesizen_util import BF16, DEVICES, F32, GPU, TARGETS
from resilient_llm_amd.engine.batch import Portion, PromptRows

D64 = torch.float64


def rel(got, want):
    got, want = got.double().cpu(), want.double()
    assert torch.isfinite(got).all()
    return float((got - want).pow(2).mean().sqrt() / want.pow(2).mean().sqrt())


def tol(dtype):
    return 3e-6 if dtype == F32 else 8e-3


def rnd(shape, seed, dtype, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * scale).to(dtype)


# ------------------------------------------------------------ streams
@pytest.mark.parametrize("device,dtype", TARGETS)
@pytest.mark.parametrize("S,W", [(1, 40), (2, 256), (3, 264), (4, 1032),
                                 (5, 2056), (6, 72), (7, 4104), (8, 128)])
def test_streams_and_norms(S, W, device, dtype):
    T, V, eps = 5, 11, 3e-4
    table = rnd((V, W), 1, dtype, 0.05)      # small: eps must matter
    ids = torch.tensor([3, 0, 10, 3, 7], dtype=torch.int32)
    we, g1, g2 = (1 + rnd((W,), s, F32, 0.3) for s in (2, 3, 4))
    inw, outw = rnd((S,), 5, F32), rnd((S,), 6, F32)
    in2 = rnd((S,), 7, F32)
    mix = rnd((S, S), 8, F32)
    x = torch.empty(T, S, W, dtype=F32, device=device)

    def dev(t):
        return t.to(device)
    h = ops.hyper_embed(dev(ids), dev(table), dev(we), x, dev(inw), dev(g1),
                        eps)
    e = plain.norm_around_zero(table.double()[ids.long()], we.double() - 1,
                               eps)
    streams = [e.clone() for _ in range(S)]
    assert rel(x, torch.stack(streams, 1)) < 3e-6
    assert rel(h, plain.norm_around_zero(
        plain.widen(streams, inw.double()), g1.double() - 1, eps)) < tol(dtype)
    for parts in (1, 3):
        y = rnd((T, parts, W), 9 + parts, dtype)
        yy = y if parts > 1 else y[:, 0].contiguous()
        rows = torch.tensor([4, 1])
        streams2 = plain.remix(streams, y.double().sum(1), mix.double(),
                               outw.double())
        last = ops.hyper_step(x, dev(yy), dev(mix), dev(outw), None, dev(g2),
                              eps, dev(rows), keep=False)
        assert rel(last, plain.norm_around_zero(
            sum(streams2), g2.double() - 1, eps)[rows]) < tol(dtype)
        assert rel(x, torch.stack(streams, 1)) < 3e-6      # left alone
        h = ops.hyper_step(x, dev(yy), dev(mix), dev(outw), dev(in2), dev(g2),
                           eps)
        streams = streams2
        assert rel(x, torch.stack(streams, 1)) < 3e-6
        assert rel(h, plain.norm_around_zero(
            plain.widen(streams, in2.double()), g2.double() - 1,
            eps)) < tol(dtype)


@pytest.mark.parametrize("device,dtype", TARGETS)
def test_relu2(device, dtype):
    x = rnd((7, 133), 1, dtype)
    want = torch.relu(x.double()) ** 2
    assert rel(ops.relu2(x.to(device)), want) < tol(dtype)


# ------------------------------------------------- windowed attention
class Attn:
    """A paged cache with scattered, poisoned pages and the op calls."""

    def __init__(self, T, H, G, dim, vdim, rot, window, keep, device, dtype,
                 base=100.0, scale=None, seed=0, cache_dtype=None):
        self.H, self.G, self.dim, self.vdim = H, G, dim, vdim
        self.window, self.keep = window, keep
        self.device, self.dtype = device, dtype
        self.rot, self.base = rot, base
        self.scale = dim ** -0.5 if scale is None else scale
        self.q, self.k = rnd((T, H, dim), seed, dtype), \
            rnd((T, G, dim), seed + 1, dtype)
        self.v = rnd((T, G, vdim), seed + 2, dtype)
        self.sink = rnd((H,), seed + 3, F32, 2.0)
        self.cs = ops.build_cos_sin(T + 1, rot, base, device=device)
        n = -(-T // 16)
        perm = torch.randperm(n + 3, generator=torch.Generator()
                              .manual_seed(seed))[:n]
        self.table = perm.to(torch.int32)[None].contiguous().to(device)
        cd = cache_dtype or dtype
        self.kc = torch.full((n + 3, G, 16, dim), float("nan")).to(cd) \
            .to(device)
        self.vc = torch.full((n + 3, G, 16, vdim), float("nan")).to(cd) \
            .to(device)

    def slots(self, p0, n):
        p = torch.arange(p0, p0 + n)
        t = self.table[0].cpu()[p // 16].long()
        return (t * 16 + p % 16).to(torch.int32).to(self.device)

    def qkv(self, p0, n, has_kv=True):
        parts = [self.q[p0:p0 + n].reshape(n, -1)]
        if has_kv:
            parts += [self.k[p0:p0 + n].reshape(n, -1),
                      self.v[p0:p0 + n].reshape(n, -1)]
        return torch.cat(parts, 1).contiguous().to(self.device)

    def run(self, p0, n, decode=False, has_kv=True, sink=True):
        pos = torch.arange(p0, p0 + n, dtype=torch.int32, device=self.device)
        args = (self.sink.to(self.device) if sink else None, self.scale,
                self.H, self.window, self.keep, has_kv)
        if decode:
            return ops.window_decode(
                self.qkv(p0, n, has_kv), self.kc, self.vc, pos, self.cs,
                self.slots(p0, n), self.table.expand(n, -1).contiguous(),
                *args)
        return ops.window_prefill(
            self.qkv(p0, n, has_kv), self.kc, self.vc, pos, self.cs,
            self.slots(p0, n), self.table,
            PromptRows([Portion(0, p0, n, 0)], self.device), *args)

    def want(self, sink=True):
        T = self.q.shape[0]
        pos = torch.arange(T)
        q, k = (plain.rotate_interleaved(t.double(), pos, self.rot, self.base)
                for t in (self.q, self.k))
        s = self.sink.double() if sink else torch.full((self.H,), -1e9,
                                                       dtype=D64)
        return plain.attend(q, k, self.v.double(), self.scale, self.window,
                            self.keep, s).reshape(T, -1)


SHAPES = [(3, 1, 20, 28, 6), (2, 2, 8, 8, 8), (4, 2, 32, 16, 16),
          (8, 2, 64, 64, 64), (6, 2, 88, 96, 16), (5, 1, 40, 72, 20),
          (7, 1, 128, 128, 64), (9, 1, 48, 48, 0), (2, 1, 136, 192, 32),
          (1, 1, 200, 256, 2), (12, 1, 16, 24, 4)]


@pytest.mark.parametrize("device,dtype", TARGETS)
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_attention_sizes(shape, device, dtype):
    H, G, dim, vdim, rot = shape
    T = 75
    a = Attn(T, H, G, dim, vdim, rot, 30, 3, device, dtype, seed=dim)
    want = a.want()
    got = torch.cat([a.run(0, 41), a.run(41, 1, decode=True), a.run(42, 2),
                     a.run(44, T - 44)])
    assert rel(got, want) < tol(dtype)
    # another layer's cached keys: same queries, other mask, no append
    a.window, a.keep = 11, 1
    want = a.want()
    got = torch.cat([a.run(0, 40, has_kv=False),
                     a.run(40, 1, decode=True, has_kv=False),
                     a.run(41, T - 41, has_kv=False)])
    assert rel(got, want) < tol(dtype)


@pytest.mark.parametrize("device,dtype", TARGETS)
@pytest.mark.parametrize("window,keep", [(1, 0), (1, 1), (2, 5), (16, 0),
                                         (17, 4), (40, 16), (64, 17),
                                         (100, 0), (10**9, 3), (5, 10**6)])
@pytest.mark.parametrize("dim", [32, 12])
def test_attention_edges_show(dim, window, keep, device, dtype):
    """Every key in turn could be the loud one: keys are one-hot loud for
    the queries at fixed distances, so a key that is let in or left out by
    one position changes the output at order one.  Prompt and decode."""
    T, H, G = 160, 2, 1
    a = Attn(T, H, G, dim, dim, 0, window, keep, device, dtype)
    a.q = torch.ones(T, H, dim).to(dtype)
    base = torch.full((T, G, dim), -0.2)
    loud = [0, keep - 1, keep, 15, 16, 63, 64]
    for i in (90, 128, 159):
        loud += [i - window, i - window + 1, i]
    for j in loud:
        if 0 <= j < T:
            base[j] = 3.0
    a.k = base.to(dtype)
    a.scale = 0.25
    a.sink = torch.tensor([2.0, -3.0])
    want = a.want()
    got = a.run(0, T)
    assert rel(got, want) < tol(dtype)
    # decode at and around the edges, over the cache the prompt wrote
    for i in (0, 1, 15, 16, 17, 63, 64, 65, 89, 90, 91, 127, 128, 129, 159):
        d = a.run(i, 1, decode=True)
        assert rel(d, want[i:i + 1]) < tol(dtype), i
    # portions that start and end at odd places
    for p0, n in ((89, 2), (90, 3), (64, 1), (63, 2), (100, 60)):
        assert rel(a.run(p0, n), want[p0:p0 + n]) < tol(dtype), (p0, n)


@pytest.mark.parametrize("device,dtype", TARGETS)
def test_sink_takes_its_share(device, dtype):
    a = Attn(50, 4, 2, 32, 32, 32, 20, 2, device, dtype, scale=0.05)
    a.sink = torch.tensor([8.0, 0.0, -5.0, 3.0])
    got = torch.cat([a.run(0, 30), *[a.run(i, 1, decode=True)
                                     for i in range(30, 50)]])
    assert rel(got, a.want()) < tol(dtype)
    norms = got.float().view(50, 4, 32).norm(dim=-1)[20:].mean(0)
    assert norms[0] < 0.05 * norms[2]         # a loud sink mutes its head
    assert rel(a.run(0, 50, sink=False), a.want(sink=False)) < tol(dtype)


@pytest.mark.parametrize("device,dtype", TARGETS)
def test_rotation_far_out(device, dtype):
    """Long positions, a large base, an outsized single score."""
    T = 700
    a = Attn(T, 2, 1, 32, 16, 32, 650, 8, device, dtype, base=1e6)
    a.k[3] *= 6
    a.k[40] *= 6
    want = a.want()
    assert rel(a.run(0, T), want) < tol(dtype)
    for i in (300, 648, 690, 699):
        assert rel(a.run(i, 1, decode=True), want[i:i + 1]) < tol(dtype)


@GPU
def test_decode_batches_and_splits():
    """Many sequences in one decode launch, few enough for key splits and
    enough for none, lengths from 1 up."""
    for B in (1, 3, 40, 300):
        lens = [1 + (37 * b) % 90 for b in range(B)]
        a = Attn(90, 8, 2, 64, 64, 32, 70, 4, "cuda:0", BF16)
        a.run(0, 90)
        want = a.want()
        n = 6                                   # pages of a sequence
        kc = a.kc[a.table[0].long()].repeat(B, 1, 1, 1)
        vc = a.vc[a.table[0].long()].repeat(B, 1, 1, 1)
        pos = torch.tensor(lens, dtype=torch.int32) - 1
        tab = torch.arange(B * n, dtype=torch.int32).view(B, n)
        slots = tab[torch.arange(B), pos.long() // 16] * 16 + pos % 16
        qkv = torch.cat([a.qkv(int(p), 1) for p in pos])
        got = ops.window_decode(
            qkv, kc, vc, pos.cuda(), a.cs, slots.to(torch.int32).cuda(),
            tab.cuda(), a.sink.cuda(), a.scale, 8, 70, 4, True)
        assert rel(got, want[pos.long()]) < tol(BF16), B


@GPU
@pytest.mark.parametrize("H,G,dim", [(8, 2, 128), (4, 2, 64), (2, 2, 128)])
@pytest.mark.parametrize("window,keep", [(1000, 40), (64, 4), (33, 0)])
def test_decode_units(H, G, dim, window, keep):
    """Windows and kept tokens that begin and end where units of 32 tokens, waves
    and parts of a sequence do; pages of 16 and of 48 tokens."""
    T = 1345
    a = Attn(T, H, G, dim, dim, 32, window, keep, "cuda:0", BF16)
    a.run(0, T)
    want = a.want()
    at = [0, 1, 31, 32, 33, 63, 64, 383, 384, 999, 1000, 1031, 1063, 1064, 1343,
          T - 1]
    for i in at:
        assert rel(a.run(i, 1, decode=True), want[i:i + 1]) < tol(BF16), i
    # pages three times as long, all of the sequence in a row
    n = -(-T // 48)
    pages = [torch.full((n, G, 48, dim), float("nan"), dtype=BF16,
                        device="cuda:0") for _ in "kv"]
    for to, src in zip(pages, (a.kc, a.vc)):
        flat = src[a.table[0].long()].transpose(0, 1).flatten(1, 2)
        for b in range(n):
            part = flat[:, b * 48:(b + 1) * 48]
            to[b, :, :part.shape[1]] = part
    table = torch.arange(n, dtype=torch.int32, device="cuda:0")[None]
    for i in at:
        pos = torch.tensor([i], dtype=torch.int32, device="cuda:0")
        got = ops.window_decode(
            a.qkv(i, 1), *pages, pos, a.cs, pos, table,
            a.sink.to("cuda:0"), a.scale, H, window, keep, True)
        assert rel(got, want[i:i + 1]) < tol(BF16), i


@GPU
@pytest.mark.parametrize("cache", [BF16, torch.float8_e4m3fn])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("H,G", [(8, 2), (4, 2), (2, 2)])
@pytest.mark.parametrize("copies", [1, 3, 9])
def test_units_of_batches(H, G, dim, cache, copies):
    """Sequences that end where units of 32 tokens, rounds of twelve and parts do,
    in batches for which they or lane groups are the faster way; against attention
    over what the cache holds."""
    T, window, keep, n = 1345, 1000, 40, 85
    a = Attn(T, H, G, dim, dim, 32, window, keep, "cuda:0", BF16,
             cache_dtype=cache)
    a.run(0, T)
    pos = torch.tensor([0, 1, 31, 32, 63, 64, 383, 384, 767, 768, 999, 1000, 1063,
                        1064, 1343, 1344] * copies, dtype=torch.int32)
    B = len(pos)
    kc, vc = (t[a.table[0].long()].repeat(B, 1, 1, 1) for t in (a.kc, a.vc))
    table = torch.arange(B * n, dtype=torch.int32).view(B, n)
    slots = table[torch.arange(B), pos.long() // 16] * 16 + pos % 16
    got = ops.window_decode(
        torch.cat([a.qkv(int(p), 1) for p in pos]), kc, vc, pos.cuda(), a.cs,
        slots.cuda(), table.cuda(), a.sink.cuda(), a.scale, H, window, keep, True)
    q = plain.rotate_interleaved(a.q.double(), torch.arange(T), 32, a.base)
    k, v = (t.view(B, n, G, 16, dim).transpose(2, 3).flatten(1, 2).float().cpu()
            .double() for t in (kc, vc))
    at = torch.arange(T)
    want = []
    for b, p in enumerate(pos.tolist()):
        seen = ((p - at < window) | (at < keep))[:p + 1]
        keys, values = (t[b, :p + 1][seen].repeat_interleave(H // G, 1)
                        for t in (k, v))
        s = torch.cat([(keys * q[p]).sum(-1) * a.scale, a.sink.double()[None]])
        want.append((torch.softmax(s, 0)[:-1, :, None] * values).sum(0).flatten())
    assert rel(got, torch.stack(want)) < tol(BF16)


@GPU
@pytest.mark.parametrize("H,G,dim", [(8, 2, 128), (4, 2, 64), (2, 2, 128)])
@pytest.mark.parametrize("window,keep", [(1000, 40), (33, 0)])
def test_newest_value_infinite(H, G, dim, window, keep):
    """An infinite value makes its channel so also as the newest token's, wherever
    in a unit of 32 tokens that is."""
    a = Attn(430, H, G, dim, dim, 32, window, keep, "cuda:0", BF16)
    inf = float("inf")
    rest = [d for d in range(dim) if d not in (7, dim - 1)]
    for i in (0, 1, 14, 30, 31, 32, 45, 399, 429):
        a.v[i, :, 7], a.v[i, :, -1] = inf, -inf
        a.run(0, i + 1)
        got, want = (t[-1].float().cpu().view(H, dim)
                     for t in (a.run(i, 1, decode=True), a.want()[:i + 1]))
        assert (got[:, 7] == inf).all() and (got[:, -1] == -inf).all(), i
        assert rel(got[:, rest], want[:, rest]) < tol(BF16), i
        a.v[i, :, 7] = a.v[i, :, -1] = 0


@GPU
def test_fp8_cache():
    a = Attn(120, 8, 2, 64, 64, 32, 50, 4, "cuda:0", BF16,
             cache_dtype=torch.float8_e4m3fn)
    got = torch.cat([a.run(0, 100), *[a.run(i, 1, decode=True)
                                      for i in range(100, 120)]])
    want = a.want()
    assert rel(got, want) < 0.08


# ----------------------------------------------- gated linear attention
def gla_case(T, H, dim, vdim, rank, tau, bias, seed, dtype):
    proj = rnd((T, 2 * H * (dim + vdim) + rank), seed, dtype)
    a2 = rnd((H * dim, rank), seed + 1, dtype, rank ** -0.5)
    b = bias + rnd((H * dim,), seed + 2, F32)
    norm = 1 + rnd((vdim,), seed + 3, F32, 0.3)
    q, k, v, g, a1 = torch.split(
        proj.double(), [H * dim, H * dim, H * vdim, H * vdim, rank], 1)
    alpha = torch.exp(torch.nn.functional.logsigmoid(
        a1 @ a2.double().T + b.double()) / tau).view(T, H, dim)
    o, S = plain.recur(q.view(T, H, dim) * dim ** -0.5, k.view(T, H, dim),
                       v.view(T, H, vdim), alpha)
    eps = 1e-3
    g = g.view(T, H, vdim)
    want = plain.rms(o, eps) * norm.double() * g * torch.sigmoid(g)
    return proj, a2, b, norm, eps, want.reshape(T, -1), S


GLA = [
    # T, heads, dim, vdim, rank, tau, bias: slow decays
    (150, 2, 40, 64, 12, 12.0, 2.0), (70, 3, 20, 18, 5, 8.0, 0.0),
    (130, 1, 128, 256, 16, 16.0, 1.0), (97, 2, 72, 30, 33, 4.0, -1.0),
    (66, 1, 256, 40, 8, 16.0, 0.0), (65, 2, 16, 16, 1, 1.0, 4.0),
    # steep: a sub-chunk decays by e^-40 and far more
    (140, 2, 32, 32, 8, 1.0, -4.0), (100, 2, 48, 20, 8, 0.25, -6.0),
    (90, 1, 64, 64, 8, 0.05, 0.0),
]


@pytest.mark.parametrize("device,dtype", TARGETS)
@pytest.mark.parametrize("case", GLA, ids=str)
def test_gla(case, device, dtype):
    T, H, dim, vdim, rank, tau, bias = case
    # exponents are differences of running log-decays: where those run
    # into the hundreds per sub-chunk, their rounding is what is left
    stol = 1e-5 if tau >= 1 else 5e-5
    proj, a2, b, norm, eps, want, S = gla_case(T, H, dim, vdim, rank, tau,
                                               bias, dim + T, dtype)
    proj, a2, b, norm = (t.to(device) for t in (proj, a2, b, norm))

    def start():
        # a used slot: what the last owner left must not be seen
        return torch.full((3, H, dim, -(-vdim // 4) * 4), float("nan"),
                          device=device)

    def prompt(state, p0, n, slot=2):
        return ops.gla_prefill(
            proj[p0:p0 + n].contiguous(), a2, b, norm, state,
            PromptRows([Portion(0, p0, n, 0, slot)], device), vdim, tau, eps)

    def token(state, p):
        return ops.gla_decode(
            proj[p:p + 1].contiguous(), a2, b, norm, state,
            torch.tensor([2], dtype=torch.int32, device=device),
            torch.tensor([p], dtype=torch.int32, device=device), vdim, tau,
            eps)

    st = start()
    assert rel(prompt(st, 0, T), want) < max(tol(dtype), stol if tau < 1 else 0)
    assert rel(st[2, :, :, :vdim], S) < stol
    st = start()
    got = torch.cat([token(st, p) for p in range(T)])
    assert rel(got, want) < max(tol(dtype), stol if tau < 1 else 0)
    assert rel(st[2, :, :, :vdim], S) < stol
    st = start()
    got, p = [], 0
    for n in [2, 17, 1, 3, 15, 16, 1, T - 55]:
        got.append(token(st, p) if n == 1 else prompt(st, p, n))
        p += n
    assert rel(torch.cat(got), want) < max(tol(dtype), stol if tau < 1 else 0)
    assert rel(st[2, :, :, :vdim], S) < stol
    assert torch.isnan(st[:2]).all()           # other slots untouched


@pytest.mark.parametrize("device,dtype", TARGETS)
def test_gla_unequal_sequences_in_one_launch(device, dtype):
    H, dim, vdim, rank, tau = 2, 32, 48, 8, 6.0
    lens = [70, 1, 129, 64, 3]
    cases = [gla_case(n, H, dim, vdim, rank, tau, 1.0, 5, dtype)
             for n in lens]
    _, a2, b, norm, eps, _, _ = cases[0]
    portions, row = [], 0
    for i, n in enumerate(lens):
        portions.append(Portion(row, 0, n, i, len(lens) - 1 - i))
        row += n
    # the decay weights of every case are the same draw
    proj = torch.cat([c[0] for c in cases]).to(device)
    st = torch.full((len(lens), H, dim, vdim), float("nan"), device=device)
    got = ops.gla_prefill(proj, a2.to(device), b.to(device), norm.to(device),
                          st, PromptRows(portions, device), vdim, tau, eps)
    row = 0
    for i, (n, c) in enumerate(zip(lens, cases)):
        assert rel(got[row:row + n], c[5]) < tol(dtype), n
        assert rel(st[len(lens) - 1 - i], c[6]) < 1e-5
        row += n


# ------------------------------------------------------------- experts
def moe_case(T, W, E, ff, seed, dtype, skew=0.0):
    h = rnd((T, W), seed, dtype)
    router = rnd((E, W), seed + 1, dtype, 2.0 * W ** -0.5)
    if skew:
        # everyone's favourite expert: aligned with a shared direction
        d = rnd((W,), seed + 9, dtype)
        h = (h.float() * 0.3 + d.float()).to(dtype)
        router[E - 1] = (d.float() * skew / W).to(dtype)
    gate, up = (rnd((E, ff, W), seed + s, dtype, 1.5 * W ** -0.5)
                for s in (2, 3))
    down = rnd((E, W, ff), seed + 4, dtype, ff ** -0.5)
    return h, router, gate, up, down


def pack(gate, up, down):
    E, ff, W = gate.shape
    ffp = -(-ff // 64) * 64
    w_up = torch.zeros(E, ffp // 16, 2, 16, W, dtype=gate.dtype)
    for g, t in enumerate((gate, up)):
        w_up[:, :, g] = torch.nn.functional.pad(
            t, (0, 0, 0, ffp - ff)).view(E, ffp // 16, 16, W)
    return w_up, torch.nn.functional.pad(down, (0, ffp - ff)).contiguous()


@pytest.mark.parametrize("device,dtype", TARGETS)
@pytest.mark.parametrize("T,W,E,top,ff,skew", [
    (1, 64, 4, 1, 64, 0), (5, 72, 5, 3, 40, 0), (33, 128, 8, 2, 96, 0),
    (64, 256, 40, 8, 64, 0), (7, 64, 3, 3, 16, 0), (50, 64, 130, 2, 32, 0),
    (300, 128, 4, 2, 80, 0), (260, 64, 6, 1, 64, 4.0),
    (1500, 64, 5, 3, 64, 0), (2100, 128, 9, 2, 200, 0),
    (30, 1088, 20, 4, 192, 0)])
def test_experts(T, W, E, top, ff, skew, device, dtype):
    limit = 0.8
    h, router, gate, up, down = moe_case(T, W, E, ff, T + E, dtype, skew)
    w_up, w_down = pack(gate, up, down)
    dev = [t.to(device) for t in (h, router, w_up, w_down)]
    ids, wts = (t.cpu() for t in ops.moe_route(dev[0], dev[1], top))
    s = torch.sigmoid(h.double() @ router.double().T)
    assert (ids.sort(1).values.diff(dim=1) > 0).all() if top > 1 else True
    assert torch.allclose(wts.double(), s.gather(1, ids.long()), atol=1e-5)
    # the chosen ones are the largest (up to exact ties)
    rest = s.scatter(1, ids.long(), -1.0).max(1).values if top < E \
        else torch.zeros(T, dtype=D64)
    assert (wts.double().min(1).values >= rest - 1e-6).all()
    if skew:
        assert (ids == E - 1).any(1).float().mean() > 0.95
    got = ops.moe_experts(*dev, top, limit).cpu()
    want = torch.zeros(T, W, dtype=D64)
    parts = torch.zeros(T, top, W, dtype=D64)
    for e in range(E):
        t, c = torch.nonzero(ids == e, as_tuple=True)
        if len(t):
            parts[t, c] = plain.clamped_expert(
                s[t, e][:, None] * h[t].double(), gate[e].double(),
                up[e].double(), down[e].double(), limit)
    want = parts.sum(1)
    assert rel(got, parts) < tol(dtype)
    assert rel(got.double().sum(1), want) < tol(dtype)


@GPU
@pytest.mark.parametrize("T,E,top,ff", [
    # rows an expert: below and above the line to tiles, low tiles alone, tiles of
    # 128 rows, low ones behind full ones and last
    (63, 4, 1, 64), (64, 4, 1, 64), (100, 4, 1, 1100), (449, 4, 1, 64),
    (452, 4, 1, 64), (300, 1, 1, 2000), (560, 2, 1, 64), (1280, 3, 1, 130),
    (700, 2, 2, 200)])
def test_heights_of_tiles(T, E, top, ff):
    test_experts(T, 64, E, top, ff, 0, "cuda:0", BF16)


@GPU
@pytest.mark.parametrize("T,E,top,ff,skew", [
    # few blocks of w: rows an expert below and above the lines to tiles, of 128
    # rows, all of them narrow or none, evenly and with one expert that has most
    (191, 4, 1, 64, 0), (192, 4, 1, 64, 0), (192, 4, 1, 64, 9), (152, 16, 2, 250, 0),
    (160, 16, 2, 250, 0), (320, 16, 2, 250, 9), (500, 8, 2, 1024, 0),
    (1000, 8, 2, 1024, 9), (3000, 8, 1, 1024, 0),
    # many: low tiles alone, behind full ones and last
    (127, 64, 8, 384, 0), (128, 64, 8, 384, 0), (800, 64, 8, 384, 0),
    (2400, 64, 8, 384, 0), (2400, 64, 8, 384, 9), (4000, 64, 8, 384, 0)])
def test_tiles_by_blocks(T, E, top, ff, skew):
    test_experts(T, 64, E, top, ff, skew, "cuda:0", BF16)


@GPU
@pytest.mark.parametrize("T,W,E", [
    # whole rounds of the router's loads, their rest, and neither; routes around
    # the lines between its kernels
    (1, 1024, 16), (17, 1032, 17), (15, 2048, 33), (16, 2056, 48),
    (33, 1288, 49), (5, 3072, 64), (16, 1024, 65), (3, 1000, 31)])
def test_rounds_of_the_router(T, W, E):
    test_experts(T, W, E, 3, 32, 0, "cuda:0", BF16)


@pytest.mark.parametrize("device", DEVICES)
def test_router_ties_go_to_the_lower_expert(device):
    h = torch.ones(3, 64)
    router = torch.zeros(70, 64)
    router[[66, 5, 20]] = 0.1
    ids, _ = ops.moe_route(h.to(device), router.to(device), 4)
    assert ids.tolist() == [[5, 20, 66, 0]] * 3


# -------------------------------------------------------------- sampler
@GPU
@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("B,V", [(1, 101), (3, 512), (40, 1003), (2, 40000)])
def test_sampler_dtypes_and_odd_vocabularies(B, V, dtype):
    logits = rnd((B, V), V, dtype).cuda()
    seeds = torch.arange(B, dtype=torch.int64)
    for temp in (0.0, 0.7):
        temps = torch.full((B,), temp)
        got = ops.sample(logits, temps.cuda(), seeds.cuda(), 3).cpu()
        if temp == 0:
            best = logits.float().max(1).values.cpu()
            picked = logits.float().cpu().gather(1, got.long()[:, None])[:, 0]
            assert torch.equal(picked, best)
        else:
            again = ops.sample(logits, temps.cuda(), seeds.cuda(), 3).cpu()
            assert torch.equal(got, again)
            assert int(got.min()) >= 0 and int(got.max()) < V
