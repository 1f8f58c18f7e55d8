"""The work that is measured: what a serving process has the framework do.

A pass is one step of the engine: a decode step through the captured graph
(``DecodeGraphRunner``), whole prompts through ``LLMEngine.feed``, a step of
chunked prefill beside decoding rows through ``forward_mixed``, or the
mixture-of-experts feed-forward as a model calls it.  Models are presets
and the sizes of ``bench.py``, weights are random, tokens and cached keys
and values come from the seed.
"""

from __future__ import annotations

import math

import torch

from resilient_llm_amd import ops
from resilient_llm_amd.engine import LLMEngine, PagedKVCache
from resilient_llm_amd.engine.graph import install_graph_runner
from resilient_llm_amd.models import (
    LlamaForCausalLM, NesizenConfig, build_model, get_config,
)
from resilient_llm_amd.models import nesizen

DEV = "cuda:0"
BLOCK = 16
NESIZEN = "nesizen-w2048"


# ------------------------------------------------------------------- cases
def listed() -> list:
    def case(name, kind, model, seqs, tokens, ragged=0.0, **kw):
        return {"name": name, "kind": kind, "model": model, "seqs": seqs,
                "tokens": tokens, "ragged": ragged, "kv8": False, "rows": 0,
                **kw}
    return [
        # one user of the small model: nothing but latency and launches
        case("decode 1b 1 sequence", "decode", "llama-3-1b", 1, 101),
        # one user of the flagship in a short chat
        case("decode 8b 1 sequence", "decode", "llama-3-8b", 1, 1000),
        # the serving benchmark's steady state: 64 clients, 128 + 64 tokens
        case("decode 8b 64 sequences", "decode", "llama-3-8b", 64, 192, 0.3),
        # long conversations, lengths as they come
        case("decode 8b long contexts", "decode", "llama-3-8b", 16, 4096,
             0.6),
        # the 8-bit cache of config.features.yaml, a batch that is not round
        case("decode 8b 8-bit cache", "decode", "llama-3-8b", 37, 2000, 0.5,
             kv8=True),
        # time to first token of a short question
        case("prompt 1b short", "prompt", "llama-3-1b", 1, 45),
        # the serving benchmark's burst: 64 prompts arrive together
        case("prompts 8b burst", "prompt", "llama-3-8b", 64, 128),
        # a document in the prompt
        case("prompt 8b long", "prompt", "llama-3-8b", 1, 7901),
        # a worker's ordinary step under load: a 512-token chunk of a long
        # prompt beside sequences that decode
        case("chunk 8b beside decodes", "chunk", "llama-3-8b", 24, 1500, 0.5,
             rows=512),
        # mixed layers: windowed attention and gated linear attention
        case("prompts nesizen", "prompt", NESIZEN, 4, 2048, 0.2),
        case("decode nesizen", "decode", NESIZEN, 16, 2048, 0.4),
        # the experts of the mixed designs over a prefill batch
        case("experts prompt rows", "experts", "moe-w2048", 1, 0, rows=6001),
    ]


def draw(rng) -> dict:
    """One more of the same ranges: batches of 1 to 64, contexts up to the
    models' 8192, prompt batches up to a worker's prefill budget."""
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["decode", "decode", "prompt", "prompt", "chunk",
                       "experts"])
    model = rng.choice(["llama-3-8b", "llama-3-8b", "llama-3-1b",
                        "mistral-7b"])
    out = {"kind": kind, "model": model, "seqs": 1, "tokens": 0,
           "ragged": round(rng.uniform(0.0, 0.8), 2), "kv8": False, "rows": 0}
    if kind == "experts":
        return {**out, "model": "moe-w2048", "ragged": 0.0,
                "rows": log(1, 8192)}
    if kind == "chunk":
        out["rows"] = log(16, 2048)
        out["seqs"] = rng.randint(1, 64)
        out["tokens"] = log(16, 8000 - out["rows"])
        out["seqs"] = max(1, min(out["seqs"], 65536 // out["tokens"]))
        return out
    if rng.random() < 0.25:
        out["model"] = NESIZEN
    if kind == "decode":
        out["seqs"] = log(1, 64)
        out["tokens"] = log(17, min(8000, 65536 // out["seqs"]))
        out["kv8"] = out["model"] != NESIZEN and rng.random() < 0.25
    else:
        total = log(16, 8000)
        out["seqs"] = max(1, min(64, total // log(16, 8000)))
        out["tokens"] = total // out["seqs"]
    return out


def lengths(case) -> list:
    """Tokens of each sequence, the first the longest."""
    return [max(1, int(case["tokens"] * (1 - case["ragged"]
                                         * (i * 0.61803 % 1.0))))
            for i in range(case["seqs"])]


# ------------------------------------------------------------------ inputs
def config_of(name: str):
    if name != NESIZEN:
        return get_config(name)
    # as bench.py measures it beside models of equal size
    return NesizenConfig.from_dict(
        {"width": 2048, "vocab": 65536, "streams": 2, "norm": {"eps": 1e-5},
         "layers": nesizen.hybrid_layers(
             12, 3,
             {"heads": 16, "kv_heads": 4, "dim": 128, "vdim": 128,
              "scale": 128 ** -0.5, "rot": {"dims": 64, "base": 1e6},
              "mask": {"size": 1024, "keep_first": 4}},
             {"heads": 8, "dim": 128, "vdim": 256, "tau": 16.0},
             {"kind": "dense", "ff": 6144})}, name=NESIZEN)


EXPERTS, CHOSEN, EXPERT_FF, WIDTH, LIMIT = 32, 4, 1024, 2048, 7.0


def prepare(case, seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    if case["kind"] == "experts":
        return _prepare_experts(case, gen)
    cfg = config_of(case["model"])
    if case["model"] == NESIZEN:
        model = build_model(cfg, device=DEV, dtype=torch.bfloat16, seed=seed)
    else:
        model = LlamaForCausalLM(cfg, device=DEV, dtype=torch.bfloat16,
                                 seed=seed)
        _settle(model.params)
    lens = lengths(case)
    need = [-(-n // BLOCK) for n in lens]
    if case["kind"] == "chunk":
        need.append(-(-(case["tokens"] + case["rows"]) // BLOCK))
    kv = PagedKVCache.for_model(
        cfg, sum(need) + 2, device=DEV, block_size=BLOCK,
        kv_dtype=torch.float8_e4m3fn if case["kv8"] else torch.bfloat16,
        state_slots=len(lens) + 1)
    engine = LLMEngine(model, kv, max_batch_size=len(lens),
                       max_prefill_tokens=16384, enable_prefix_caching=False)
    state = {"kind": case["kind"], "model": model, "kv": kv, "engine": engine,
             "lens": lens}

    def tokens(n):
        return torch.randint(5, cfg.vocab_size, (n,), generator=gen,
                             device=DEV, dtype=torch.int32)
    if case["kind"] == "prompt":
        ids = tokens(sum(lens)).tolist()
        state["entries"], state["names"] = [], []
        for i, n in enumerate(lens):
            state["entries"].append((f"p{i}", ids[:n], [n - 1]))
            state["names"].append(f"p{i}")
            ids = ids[n:]
        return state

    if case["kind"] == "decode":
        install_graph_runner(engine, max_blocks_per_seq=max(need))
    _fill_cache(kv, cfg, gen)
    # pages as a long-running pool hands them out: in no order
    free = torch.tensor(kv.allocate(sum(need)), dtype=torch.int32, device=DEV)
    free = free[torch.randperm(len(free), generator=gen, device=DEV)]
    tables = torch.zeros((len(need), max(need)), dtype=torch.int32,
                         device=DEV)
    at = 0
    for i, n in enumerate(need):
        tables[i, :n] = free[at:at + n]
        at += n
    last = torch.tensor(lens, dtype=torch.int32, device=DEV) - 1
    if case["kind"] == "decode":
        slots = None if kv.states is None else torch.tensor(
            [kv.states.allocate() for _ in lens], dtype=torch.int32,
            device=DEV)
        state.update(batch=(
            tokens(len(lens)), last, tables,
            torch.zeros(len(lens), device=DEV),
            torch.arange(len(lens), device=DEV), slots))
        return state

    B, n, start = len(lens), case["rows"], case["tokens"]
    pos = torch.cat([last, torch.arange(start, start + n, dtype=torch.int32,
                                        device=DEV)])
    row = torch.cat([torch.arange(B, device=DEV),
                     torch.full((n,), B, device=DEV)])
    slots = tables[row, (pos // BLOCK).long()] * BLOCK + pos % BLOCK
    tile = torch.arange(0, n, 32, dtype=torch.int32, device=DEV)
    state["args"] = (
        tokens(B + n), pos, kv, slots.int(), B, tables[:B, :max(need[:B])]
        .contiguous(), last + 1, B + tile, start + tile,
        torch.clamp(n - tile, max=32), torch.zeros_like(tile),
        tables[B:].contiguous(),
        torch.cat([torch.arange(B, device=DEV),
                   torch.tensor([B + n - 1], device=DEV)]))
    return state


def _settle(params) -> None:
    """A residual of size one to which every layer adds a tenth or so, as
    in trained models; drawn alike, weights amplify each rounding."""
    params["embed"].mul_(50.0)
    for name, w in params.items():
        if name.endswith((".o", ".down")):
            w.mul_(0.25)


def _fill_cache(kv, cfg, gen) -> None:
    """Keys, values and states of a size that projections of normed inputs
    with these weights have."""
    scale = 0.02 * cfg.hidden_size ** 0.5

    def fill(t, std):
        for part in t:
            part.copy_(torch.empty(part.shape, dtype=torch.bfloat16,
                                   device=DEV).normal_(0.0, std,
                                                       generator=gen))
    if kv.states is None:
        fill(kv.k, scale)
        fill(kv.v, scale)
        return
    for i, spec in enumerate(cfg.layers):
        if isinstance(spec.mixer, nesizen.AttentionSpec):
            for t in kv.layer(i):
                fill(t, scale)
        else:
            # outer products summed over a memory of about 125 tokens
            kv.states.layer(i).normal_(0.0, scale * scale * 63 ** 0.5,
                                       generator=gen)


def _prepare_experts(case, gen):
    def mat(*shape, std=0.02):
        return torch.empty(shape, dtype=torch.bfloat16, device=DEV).normal_(
            0.0, std, generator=gen)
    return {"kind": "experts",
            "args": (mat(case["rows"], WIDTH, std=1.0),
                     mat(EXPERTS, WIDTH),
                     mat(EXPERTS, EXPERT_FF // 16, 2, 16, WIDTH),
                     mat(EXPERTS, WIDTH, EXPERT_FF), CHOSEN, LIMIT)}


# -------------------------------------------------------------------- pass
def run(state):
    kind = state["kind"]
    if kind == "experts":
        return ops.moe_experts(*state["args"])
    if kind == "prompt":
        return {"logits": state["engine"].feed(state["entries"],
                                               end=state["names"]),
                **_held(state)}
    if kind == "decode":
        runner = state["engine"].graph_runner
        runner.load(*state["batch"])
        _, logits = runner.step()
    else:
        logits = state["model"].forward_mixed(*state["args"])
    return {"logits": logits, **_held(state)}


def _held(state) -> dict:
    """What the pass wrote besides its logits: the cache, recurrent
    states."""
    kv = state["kv"]
    if kv.states is None:
        def plain(t):
            return t.view(torch.uint8) if t.element_size() == 1 else t
        return {"keys": plain(kv.k), "values": plain(kv.v)}
    layers = state["model"].config.layers
    return {"held": [t for i, s in enumerate(layers) for t in (
        kv.layer(i) if isinstance(s.mixer, nesizen.AttentionSpec)
        else (kv.states.layer(i),))]}


# -------------------------------------------------------------------- work
def work(case) -> dict:
    if case["kind"] == "experts":
        t, picks = case["rows"], case["rows"] * CHOSEN
        used = EXPERTS * (1 - (1 - CHOSEN / EXPERTS) ** t)
        one = 3 * EXPERT_FF * WIDTH
        return {"bytes": 2 * (used * one + t * WIDTH + picks * WIDTH
                              + EXPERTS * WIDTH),
                "flops": 2 * (picks * one + t * EXPERTS * WIDTH)}
    cfg, lens = config_of(case["model"]), lengths(case)
    decode = case["kind"] == "decode"
    rows = len(lens) if decode else sum(lens)
    logit_rows = len(lens)
    if case["kind"] == "chunk":
        rows, logit_rows = len(lens) + case["rows"], len(lens) + 1
    # (query, key) pairs and cached tokens that a full-attention layer sees
    if case["kind"] == "prompt":
        pairs, cached = sum(n * (n + 1) / 2 for n in lens), 0
    else:
        pairs = cached = sum(lens)
        if case["kind"] == "chunk":
            n, start = case["rows"], case["tokens"]
            pairs += n * start + n * (n + 1) / 2
            cached += start
    d, V = cfg.hidden_size, cfg.vocab_size
    small = 1 if case["kv8"] else 2
    logits = logit_rows * V
    if case["model"] != NESIZEN:
        wide = (cfg.q_size + 2 * cfg.kv_size + cfg.q_size) * d
        ffn = 3 * cfg.intermediate_size * d
        per_token = 2 * cfg.kv_size * small
        return {
            "bytes": cfg.n_layers * (2 * (wide + ffn)
                                     + per_token * (cached + rows))
            + 2 * V * d + (2 if case["kind"] != "prompt" else 4) * logits
            + 2 * rows * d,
            "flops": 2 * rows * cfg.n_layers * (wide + ffn)
            + 2 * logits * d + 4 * cfg.n_layers * cfg.q_size * pairs}
    total, flops = 2 * V * d + 2 * rows * d + 2 * logits, 2 * logits * d
    for spec in cfg.layers:
        m = spec.mixer
        attn = isinstance(m, nesizen.AttentionSpec)
        if attn:
            seen = [min(n, m.window + m.keep_first) for n in lens]
            kv = m.kv_heads * (m.dim + m.vdim)
            w = (m.heads * (m.dim + m.vdim) + kv) * d
            total += 2 * kv * ((sum(seen) if decode else 0) + rows)
            flops += 2 * m.heads * (m.dim + m.vdim) * (
                sum(seen) if decode else sum(
                    n * s - s * (s - 1) / 2 for n, s in zip(lens, seen)))
        else:
            w = (m.heads * (2 * m.dim + 3 * m.vdim) + cfg.decay_rank) * d
            total += 4 * m.heads * m.dim * m.vdim * len(lens) * (
                2 if decode else 1)
            flops += 6 * m.heads * m.dim * m.vdim * rows
        w += 2 * spec.mlp.ff * d
        total += 2 * w
        flops += 2 * w * rows
    return {"bytes": total, "flops": flops}


def tolerance(case) -> dict:
    if case["kind"] == "experts":
        return {"rel": 0.01, "max": 0.2}
    if case["model"] == NESIZEN:
        return {"rel": 0.02, "max": 0.3}
    # the 16-bit residual is rounded twice a layer: with its products summed
    # in another order a pass came out 1.2 % off itself over 32 layers (and
    # is 1.4 % off 64 bits)
    return {"rel": 0.03, "max": 0.3, "differ": 0.005}


# ------------------------------------------------------------- in 64 bits
def exact(case, seed):
    state = prepare(case, seed)
    if case["kind"] == "experts":
        return _exact_experts(*state["args"])
    if case["model"] == NESIZEN:
        logits, held = _exact_nesizen(case, state)
        return {"logits": logits, "held": held}
    return {"logits": _exact_llama(case, state), "keys": None, "values": None}


def _rows_of(case, state):
    """(tokens, positions, [(first row, rows, first position, page table)]
    per sequence, rows whose logits are returned)."""
    if case["kind"] == "prompt":
        ids = torch.tensor([t for _, ts, _ in state["entries"] for t in ts],
                           device=DEV)
        lens, at, seqs, pos, last = state["lens"], 0, [], [], []
        for n in lens:
            seqs.append((at, n, 0, None))
            pos += range(n)
            at += n
            last.append(at - 1)
        return ids, torch.tensor(pos, device=DEV), seqs, last
    if case["kind"] == "decode":
        ids, pos, tables = state["batch"][:3]
        seqs = [(i, 1, n - 1, tables[i]) for i, n in enumerate(state["lens"])]
        return ids.long(), pos.long(), seqs, list(range(len(seqs)))
    a = state["args"]
    B = a[4]
    seqs = [(i, 1, n - 1, a[5][i]) for i, n in enumerate(state["lens"])]
    seqs.append((B, case["rows"], case["tokens"], a[11][0]))
    return a[0].long(), a[1].long(), seqs, a[12].tolist()


def _rms(x, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps)


def _turn(x, pos, freq, halves: bool):
    """x [T, heads, dim]: pairs of the first 2 len(freq) channels, (i, i +
    half) or (2 i, 2 i + 1), turned by position times frequency."""
    n = 2 * len(freq)
    ang = pos.double()[:, None, None] * freq
    c, s = ang.cos(), ang.sin()
    a, b = ((x[..., :n // 2], x[..., n // 2:n]) if halves
            else (x[..., 0:n:2], x[..., 1:n:2]))
    turned = (a * c - b * s, b * c + a * s)
    turned = (torch.cat(turned, -1) if halves
              else torch.stack(turned, -1).flatten(-2))
    return torch.cat([turned, x[..., n:]], -1)


def _cached(pages, table, n):
    """First ``n`` tokens of a sequence: [kv heads, n, dim]."""
    if not n:
        return pages.new_zeros((pages.shape[1], 0, pages.shape[3])).double()
    got = pages[table[:-(-n // BLOCK)].long()].transpose(0, 1)
    return got.reshape(pages.shape[1], -1, pages.shape[3])[:, :n] \
        .float().double()


def _attend(q, k, v, scale, pos, window=None, keep=0, sink=None):
    """q [T, H, dim] over k, v [G, n, dim] of positions 0 .. n - 1."""
    H, G = q.shape[1], k.shape[0]
    out = torch.empty((q.shape[0], H, v.shape[2]), dtype=q.dtype, device=DEV)
    at = torch.arange(k.shape[1], device=DEV)
    for r in range(0, len(q), 1024):
        p = pos[r:r + 1024, None]
        hidden = at > p
        if window is not None:
            hidden |= (p - at >= window) & (at >= keep)
        hi = int(p.max()) + 1
        for h in range(H):
            g = h // (H // G)
            s = q[r:r + 1024, h] @ k[g, :hi].T * scale
            s.masked_fill_(hidden[:, :hi], float("-inf"))
            if sink is not None:
                s = torch.cat([s, sink[h].expand(len(s), 1)], 1)
            w = torch.softmax(s, -1)[:, :hi]
            out[r:r + 1024, h] = w @ v[g, :hi]
    return out.flatten(1)


def _exact_llama(case, state):
    model, kv = state["model"], state["kv"]
    P, c = model.params, model.config
    ids, pos, seqs, wanted = _rows_of(case, state)

    def mat(name):
        return P[name].double()
    half = c.head_dim // 2
    freq = c.rope_theta ** (-torch.arange(half, dtype=torch.float64,
                                          device=DEV) / half)
    x = P["embed"][ids].double()
    for i in range(c.n_layers):
        h = _rms(x, c.rms_eps) * P[f"l{i}.ln1"].double()
        q, k, v = torch.split(h @ mat(f"l{i}.qkv").T,
                              [c.q_size, c.kv_size, c.kv_size], 1)
        q = _turn(q.reshape(len(x), c.n_heads, -1), pos, freq, True)
        k = _turn(k.reshape(len(x), c.n_kv_heads, -1), pos, freq, True)
        v = v.reshape(len(x), c.n_kv_heads, -1)
        o = torch.empty((len(x), c.q_size), dtype=x.dtype, device=DEV)
        for r, n, start, table in seqs:
            own = [t[r:r + n].transpose(0, 1) for t in (k, v)]
            keys, values = (
                torch.cat([_cached(pages, table, start), t], 1).contiguous()
                if start else t.contiguous()
                for pages, t in zip((kv.k[i], kv.v[i]), own))
            o[r:r + n] = _attend(q[r:r + n], keys, values,
                                 c.head_dim ** -0.5, pos[r:r + n])
        x = x + o @ mat(f"l{i}.o").T
        h = _rms(x, c.rms_eps) * P[f"l{i}.ln2"].double()
        g, u = (h @ mat(f"l{i}.gate_up").T).chunk(2, 1)
        x = x + (g * torch.sigmoid(g) * u) @ mat(f"l{i}.down").T
    h = _rms(x[wanted], c.rms_eps) * P["final_ln"].double()
    return h @ mat("lm_head").T


def _exact_nesizen(case, state):
    model, kv = state["model"], state["kv"]
    c = model.config
    ids, pos, seqs, wanted = _rows_of(case, state)
    P = model.params
    eps, T = c.rms_eps, len(ids)
    lens = state["lens"]
    x = (_rms(P["embed"][ids].double(), eps) * P["embed.norm"].double())
    x = x[:, None].expand(T, c.streams, -1)
    held = []

    def sublayer(x, i, q, f):
        p = {k: P[f"l{i}.hc{q}.{k}"].double() for k in ("in", "out", "mix")}
        h = (p["in"][:, None] * x).sum(1)
        y = f(_rms(h, eps) * P[f"l{i}.norm{q}"].double())
        mixed = torch.stack([(p["mix"][:, t, None] * x).sum(1)
                             for t in range(c.streams)], 1)
        return mixed + p["out"][:, None] * y[:, None]

    def attention(i, m, h):
        H, G = m.heads, m.kv_heads
        q, k, v = torch.split(h @ P[f"l{i}.proj"].double().T,
                              [H * m.dim, G * m.dim, G * m.vdim], 1)
        freq = m.rot_base ** (-2 * torch.arange(
            m.rot_dims // 2, dtype=torch.float64, device=DEV) / m.rot_dims)
        q = _turn(q.reshape(T, H, -1), pos, freq, False)
        k = _turn(k.reshape(T, G, -1), pos, freq, False)
        v = v.reshape(T, G, -1)
        o = torch.empty((T, H * m.vdim), dtype=h.dtype, device=DEV)
        for r, n, start, table in seqs:
            keys, values = (
                torch.cat([_cached(pages, table, start),
                           t[r:r + n].transpose(0, 1)], 1).contiguous()
                if start else t[r:r + n].transpose(0, 1).contiguous()
                for pages, t in zip(kv.layer(i), (k, v)))
            o[r:r + n] = _attend(q[r:r + n], keys, values, m.scale,
                                 pos[r:r + n], m.window, m.keep_first,
                                 P[f"l{i}.sink"].double())
        held.extend([None, None])
        return o @ P[f"l{i}.o"].double().T

    def recurrence(i, m, h):
        H, D, V = m.heads, m.dim, m.vdim
        q, k, v, g, a1 = torch.split(
            h @ P[f"l{i}.proj"].double().T,
            [H * D, H * D, H * V, H * V, c.decay_rank], 1)
        z = a1 @ P[f"l{i}.a2"].double().T + P[f"l{i}.a2.b"].double()
        alpha = torch.exp(torch.nn.functional.logsigmoid(z) / m.tau)
        n = max(e[1] for e in seqs)
        # sequences side by side, short ones padded with what keeps a state
        side = [torch.zeros((n, len(seqs), H, w), dtype=h.dtype, device=DEV)
                for w in (D, D, V)]
        keep = torch.ones((n, len(seqs), H, D), dtype=h.dtype, device=DEV)
        for s, (r, rows, _, _) in enumerate(seqs):
            for dst, src in zip([*side, keep], (q, k, v, alpha)):
                dst[:rows, s] = src[r:r + rows].view(rows, H, -1)
        whole = kv.states.layer(i).double()
        slots = None if case["kind"] == "prompt" \
            else state["batch"][5].long()
        S = torch.zeros((len(seqs), H, D, V), dtype=h.dtype, device=DEV)
        if slots is not None:
            fresh = pos[:, None, None, None] == 0
            S = torch.where(fresh, S, whole[slots])
        o = torch.empty((n, len(seqs), H, V), dtype=h.dtype, device=DEV)
        for t in range(n):
            S = keep[t][..., None] * S \
                + side[1][t][..., None] * side[2][t][..., None, :]
            o[t] = (side[0][t][..., None] * S).sum(-2) * D ** -0.5
        if slots is not None:
            whole[slots] = S
            held.append(whole)
        else:
            held.append(None)
        o = torch.cat([o[:rows, s] for s, (_, rows, _, _)
                       in enumerate(seqs)])
        o = _rms(o, eps) * P[f"l{i}.gla_norm"].double()
        o = o.flatten(1) * g * torch.sigmoid(g)
        return o @ P[f"l{i}.o"].double().T

    for i, spec in enumerate(c.layers):
        m = spec.mixer
        mixer = attention if isinstance(m, nesizen.AttentionSpec) \
            else recurrence
        x = sublayer(x, i, 1, lambda h: mixer(i, m, h))
        x = sublayer(x, i, 2, lambda h: torch.relu(
            h @ P[f"l{i}.up"].double().T) ** 2
            @ P[f"l{i}.down"].double().T)
    h = _rms(x[wanted].sum(1), eps) * P["final.norm"].double()
    assert len(lens) == len(seqs)
    return h @ P["head"].double().T, held


def _exact_experts(h, router, w_up, w_down, top, limit):
    x = h.double()
    s, ids = torch.sort(torch.sigmoid(x @ router.double().T), dim=-1,
                        descending=True, stable=True)
    s, ids = s[:, :top], ids[:, :top]
    y = torch.zeros((len(h), top, h.shape[1]), dtype=x.dtype, device=DEV)
    for e in range(len(router)):
        t, k = torch.nonzero(ids == e, as_tuple=True)
        rows = x[t] * s[t, k][:, None]
        up = w_up[e].double()
        gate = torch.clamp(rows @ up[:, 0].reshape(-1, h.shape[1]).T,
                           max=limit)
        u = torch.clamp(rows @ up[:, 1].reshape(-1, h.shape[1]).T, -limit,
                        limit)
        y[t, k] = (gate * torch.sigmoid(1.702 * gate) * (u + 1)) \
            @ w_down[e].double().T
    return y
