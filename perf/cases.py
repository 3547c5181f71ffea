"""The work that programs have this library do, as cases that can be timed and compared.

A case is one call, or one request's worth of calls, of the public entry points over one
configuration: decode steps and prefill / training chunks over a compressed cache, streams of
blocks committed through the flush (attach route with and without the Alpha exact pool and Beta,
unified route), streaming training, and a small served model. ``listed()`` names the usual sizes,
``draw(rng)`` picks others from the same ranges.

The configuration is the benchmark's wherever a case does not say otherwise: 12 clusters, B = 128
slots per level, mid anchors, an exact pool of 256 tokens with spans of at most 64, Beta novelty and
the 4 -> 2 merges, spans that end every 32 tokens, rows from a mixture of 12 Gaussians around
centers N(0, 1) * 4 with 10% outliers N(0, 1) * 12.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from logkv_amd import (LogKVStreamingAttention, LogKVStreamTrainingAttention, LogStructuredKVCache, flush_grouping,
                       log_kv_chunk_attention, set_flush_grouping)

K, B, EXACT, SPAN = 12, 128, 256, 64
DTYPES = {"bfloat16": torch.bfloat16, "float16": torch.float16, "float32": torch.float32}

# Buffers that a stream of commits leaves behind (the exact pool's follow when there is one).
STATE = ("level_k", "level_v", "level_w", "level_p_lo", "level_p_hi", "level_sum_wp", "level_order", "pad_mask",
         "level_count", "centroid", "n_eff", "n_total", "p_hi_c", "level0_phase", "alive", "recent_k", "recent_v",
         "recent_k_raw", "recent_pos")
ALPHA_STATE = ("alpha_k_raw", "alpha_v", "alpha_pos", "alpha_valid", "alpha_span_len", "alpha_span_closed",
               "alpha_span_count", "alpha_count_dev")


def listed():
    return [
        # One token of one short conversation: the smallest call of a serving loop, latency and launches.
        dict(name="decode_1x4k", kind="decode", batch=1, groups=8, heads=16, dim=128, context=4096, recent=512,
             rows=1, alpha=True, dtype="bfloat16"),
        # One token of each of eight 32K conversations: the benchmark's decode.
        dict(name="decode_8x32k", kind="decode", batch=8, groups=8, heads=16, dim=128, context=32768, recent=2048,
             rows=1, alpha=True, dtype="bfloat16"),
        # Eight query heads to a KV head, four 16K conversations.
        dict(name="decode_wide_4x16k", kind="decode", batch=4, groups=8, heads=64, dim=128, context=16384,
             recent=1024, rows=1, alpha=True, dtype="bfloat16"),
        # A follow-up question over a short history: an odd chunk, 64-wide heads.
        dict(name="chunk_333_d64", kind="chunk", batch=2, groups=4, heads=8, dim=64, context=4096, recent=512,
             rows=333, alpha=False, dtype="bfloat16"),
        # One layer of the streaming prefill late in a 32K prompt: a 2048-row block over its prefix.
        dict(name="chunk_2048x32k", kind="chunk", batch=1, groups=8, heads=16, dim=128, context=32768, recent=2048,
             rows=2048, alpha=True, dtype="bfloat16"),
        # A training chunk, forward and backward, over the detached prefix.
        dict(name="train_chunk_2x1024", kind="train", batch=2, groups=8, heads=16, dim=128, context=16384,
             recent=1024, rows=1024, alpha=True, dtype="bfloat16"),
        # Streaming training of one layer over a sequence: recorded forward, replayed backward.
        dict(name="train_stream_4k", kind="train_stream", batch=1, groups=8, heads=16, dim=128, tokens=4096,
             recent=512, block=512, alpha=True),
        # Short blocks into a small cache: a flush of few rows, latency and launches.
        dict(name="flush_128x12", kind="flush", batch=1, groups=4, dim=64, recent=128, blocks=12, alpha=True,
             unified=False),
        # One layer alone, attach route only: the flush of the CPU reference configuration.
        dict(name="flush_layer_2048x5", kind="flush", batch=1, groups=8, dim=128, recent=2048, blocks=5, alpha=False,
             unified=False),
        # A 28-layer model's caches flushed together as batch rows: the benchmark's flush.
        dict(name="flush_model_2048x6", kind="flush", batch=28, groups=8, dim=128, recent=2048, blocks=6, alpha=True,
             unified=False),
        # The unified route at its benchmark geometry (the first flush into empty clusters, and the next).
        dict(name="unified_4096x3", kind="flush", batch=4, groups=8, dim=128, recent=4096, blocks=3, alpha=False,
             unified=True),
        # A request served by a small model: chunked prefill through every layer, then decode steps.
        dict(name="serve_5001", kind="serve", layers=4, groups=8, heads=16, dim=128, recent=1024, prompt=5001,
             decode=12),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("decode", "decode", "chunk", "chunk", "train", "flush", "flush", "unified"))
    alpha = rng.random() < 0.6
    if kind in ("decode", "chunk", "train"):
        dim = rng.choice((64, 96, 128, 128))
        groups = rng.choice((2, 4, 8))
        per_group = rng.choice((1, 2, 2, 3, 4, 5, 8)) if kind == "decode" else rng.choice((1, 2, 3, 4))
        recent = 2 * _log_uniform(rng, 64, 1024)
        context = max(recent + EXACT + K, _log_uniform(rng, 2048, 32768))
        batch = _log_uniform(rng, 1, 16 if kind == "decode" else 2)
        rows = {"decode": rng.choice((1, 1, 1, 2)), "chunk": _log_uniform(rng, 17, recent),
                "train": _log_uniform(rng, 17, min(recent, 1024))}[kind]
        dtype = rng.choice(("bfloat16", "bfloat16", "bfloat16", "float16", "float32"))
        return dict(kind=kind, batch=batch, groups=groups, heads=groups * per_group, dim=dim, context=context,
                    recent=recent, rows=rows, alpha=alpha, dtype=dtype)
    if kind == "flush":
        return dict(kind="flush", batch=_log_uniform(rng, 1, 28), groups=rng.choice((2, 4, 8)),
                    dim=rng.choice((64, 128, 128, 192)), recent=_log_uniform(rng, 64, 2048), blocks=rng.randint(3, 6),
                    alpha=alpha, unified=False)
    return dict(kind="flush", batch=_log_uniform(rng, 1, 4), groups=rng.choice((2, 4, 8)), dim=rng.choice((64, 128)),
                recent=_log_uniform(rng, 256, 4096), blocks=3, alpha=False, unified=True)


# ----------------------------------------------------------------------
# Inputs
# ----------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(shape, g):
    return torch.randn(shape, generator=g, device="cuda")


def _mixture(batch, groups, rows, dim, g):
    """Rows around 12 centers, 10% far outliers, bf16 ``[batch, groups, rows, dim]``."""
    out = torch.empty(batch, groups, rows, dim, dtype=torch.bfloat16, device="cuda")
    for b in range(batch):
        centers = _randn((groups, 12, dim), g) * 4.0
        label = torch.randint(0, 12, (groups, rows), generator=g, device="cuda")
        x = torch.gather(centers, 1, label[..., None].expand(-1, -1, dim)) + _randn((groups, rows, dim), g) * 0.5
        far = torch.rand(groups, rows, generator=g, device="cuda") < 0.1
        out[b] = torch.where(far[..., None], _randn((groups, rows, dim), g) * 12.0, x)
    return out


def _tables(positions, dim):
    """Rotate-half RoPE tables, float32 ``[positions, dim]``."""
    theta = 1.0 / (10000.0 ** (torch.arange(0, dim, 2, dtype=torch.float32, device="cuda") / dim))
    angle = torch.outer(torch.arange(positions, dtype=torch.float32, device="cuda"), theta)
    angle = torch.cat((angle, angle), dim=-1)
    return torch.cos(angle), torch.sin(angle)


def _rope(x, cos, sin):
    half = x.size(-1) // 2
    return x * cos + torch.cat((-x[..., half:], x[..., :half]), dim=-1) * sin


def _span_ends(batch, tokens):
    at = torch.arange(tokens, device="cuda")[None, :] + 7 * torch.arange(batch, device="cuda")[:, None]
    return (at % 32 == 0).to(torch.uint8)


def _cache(batch, groups, dim, max_seq, recent, alpha, unified=False, replay=False, grouped=False):
    cos, sin = _tables(max_seq, dim)
    before = flush_grouping()
    set_flush_grouping(grouped)
    try:
        return LogStructuredKVCache(
            (batch, groups, max_seq, dim), (batch, groups, max_seq, dim), B=B, recent_size=recent, device="cuda",
            dtype=torch.bfloat16, semantic_clusters=True, cluster_k_max=K, semantic_s_h=0.5 * dim,
            semantic_flush_granularity=recent, semantic_anchor_mode="mid", allocate_second_order=False,
            semantic_unified_route=unified, semantic_replay_updates=replay, cos_cache=cos, sin_cache=sin,
            rope_n_elem=dim, alpha_exact_tokens=EXACT if alpha else 0, alpha_span_max_tokens=SPAN,
            beta_novelty=alpha, beta_adaptive_merge=alpha)
    finally:
        set_flush_grouping(before)


def _fenwick_counts(share, flushes, slots, levels):
    """Slots in use per level of ladders that took ``share`` rows each over ``flushes`` flushes."""
    left = share.copy()
    chunk = np.maximum(1, share // flushes)
    counts = np.zeros((levels, share.size), dtype=np.int64)
    while left.any():
        m = np.minimum(chunk, left)
        left -= m
        for level in range(levels):
            rest = m - np.minimum(slots - counts[level], m)
            carry = np.zeros_like(rest) if level == levels - 1 else (rest + 1) // 2
            counts[level] = np.where(rest > 0, slots if level == levels - 1 else slots + rest - 2 * carry,
                                     counts[level] + m)
            m = carry
    return counts


def _levels(case):
    """(slots per level, levels) of the case's cache, as its constructor sizes them."""
    from logkv_amd import ladder_budget
    return ladder_budget(case["batch"], case["groups"], case["context"], case["dim"], case["dim"], B, K,
                         EXACT if case["alpha"] else 0, 2)[:2]


def _slot_counts(case, share):
    slots, levels = _levels(case)
    return _fenwick_counts(share.reshape(-1), 15, slots, levels).T.reshape(*share.shape, levels)


def _archived(case):
    return case["context"] - case["recent"] - (EXACT if case["alpha"] else 0)


def _readout_state(case, seed):
    """A compressed cache late in a conversation: occupied slots with masses in [1, 64) and anchors in the
    archived part, a full exact pool (5% of its rows invalid) and a full recent window."""
    g = _gen(seed)
    batch, groups, dim, recent = case["batch"], case["groups"], case["dim"], case["recent"]
    slots, levels = _levels(case)
    rng = np.random.default_rng(seed)
    share = rng.random((batch, groups, K)) + 0.5
    share = (share / share.sum(-1, keepdims=True) * _archived(case)).astype(np.int64)
    counts = torch.from_numpy(_slot_counts(case, share)).cuda()
    used = torch.arange(slots, device="cuda") < counts[..., None]
    shape = (batch, groups, K, levels, slots)
    horizon = max(_archived(case), 1)
    w = (torch.rand(shape, generator=g, device="cuda") * 63 + 1).floor() * used
    anchor = torch.randint(0, horizon, shape, generator=g, device="cuda")
    bf = torch.bfloat16
    state = {"level_count": counts.to(torch.int16), "level_w": w, "level_sum_wp": w.long() * anchor,
             "level_k": (_randn((*shape, dim), g) * used[..., None]).to(bf),
             "level_v": (_randn((*shape, dim), g) * used[..., None]).to(bf),
             "recent_k": _randn((batch, groups, recent, dim), g).to(bf),
             "recent_v": _randn((batch, groups, recent, dim), g).to(bf)}
    if case["alpha"]:
        state["alpha_k_raw"] = _randn((batch, groups, EXACT, dim), g).to(bf)
        state["alpha_v"] = _randn((batch, groups, EXACT, dim), g).to(bf)
        state["alpha_pos"] = torch.randint(0, horizon, (batch, EXACT), generator=g, device="cuda")
        state["alpha_valid"] = torch.rand(batch, EXACT, generator=g, device="cuda") < 0.95
    dtype = DTYPES[case["dtype"]]
    rows = {n: _randn((batch, h, case["rows"], dim), g).to(dtype)
            for n, h in (("q", case["heads"]), ("k", groups), ("v", groups), ("dout", case["heads"]))}
    return state, rows


def _filled_cache(case, state):
    cache = _cache(case["batch"], case["groups"], case["dim"], case["context"], case["recent"], case["alpha"])
    for name, t in state.items():
        dst = getattr(cache, name)
        (dst[:, :, :case["recent"]] if name.startswith("recent") else dst).copy_(t)
    cache.recent_count = case["recent"]
    if case["alpha"]:
        cache.alpha_count = EXACT
    cache.token_count = _archived(case) + case["recent"]
    return cache


def _stream_rows(batch, groups, tokens, dim, cos, sin, g):
    """(post-RoPE keys, values, pre-RoPE keys) of a stream, bf16."""
    k_raw = _mixture(batch, groups, tokens, dim, g)
    v = _randn((batch, groups, tokens, dim), g).to(torch.bfloat16)
    k = torch.empty_like(k_raw)
    for b in range(batch):
        k[b] = _rope(k_raw[b].float(), cos[:tokens], sin[:tokens])
    return k, v, k_raw


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("decode", "chunk", "train"):
        state, rows = _readout_state(case, seed)
        if kind == "train":
            for n in ("q", "k", "v"):
                rows[n].requires_grad_(True)
        return dict(case=case, cache=_filled_cache(case, state), **rows)
    g = _gen(seed)
    if kind == "flush":
        tokens = case["recent"] * case["blocks"]
        cache = _cache(case["batch"], case["groups"], case["dim"], tokens, case["recent"], case["alpha"],
                       case["unified"])
        k, v, k_raw = _stream_rows(case["batch"], case["groups"], tokens, case["dim"], cache.cos_cache,
                                   cache.sin_cache, g)
        return dict(case=case, cache=cache, k=k, v=v, k_raw=k_raw, pos=torch.arange(tokens, device="cuda"),
                    ends=_span_ends(case["batch"], tokens) if case["alpha"] else None)
    if kind == "train_stream":
        tokens, batch = case["tokens"], case["batch"]
        cache = _cache(batch, case["groups"], case["dim"], tokens, case["recent"], case["alpha"], replay=True)
        k, v, k_raw = _stream_rows(batch, case["groups"], tokens, case["dim"], cache.cos_cache, cache.sin_cache, g)
        q = _randn((batch, case["heads"], tokens, case["dim"]), g).to(torch.bfloat16)
        dout = _randn(q.shape, g).to(torch.bfloat16)
        ends = _span_ends(batch, tokens).cpu().tolist() if case["alpha"] else None
        return dict(case=case, cache=cache, q=q.requires_grad_(True), k=k.requires_grad_(True),
                    v=v.requires_grad_(True), k_raw=k_raw, dout=dout, ends=ends)
    # A server: one cache and engine per layer, warmed up by a request long enough to flush.
    tokens, recent = case["prompt"] + case["decode"], case["recent"]
    max_seq = (tokens // recent + 2) * recent
    caches = [_cache(1, case["groups"], case["dim"], max_seq, recent, True, grouped=True)
              for _ in range(case["layers"])]
    engines = [LogKVStreamingAttention(c, case["dim"] ** -0.5, prefill_block=recent) for c in caches]
    layers = []
    for c in caches:
        k, v, k_raw = _stream_rows(1, case["groups"], tokens, case["dim"], c.cos_cache, c.sin_cache, g)
        q = _rope(_randn((1, case["heads"], tokens, case["dim"]), g), c.cos_cache[:tokens], c.sin_cache[:tokens])
        layers.append((q.to(torch.bfloat16), k, v, k_raw))
    state = dict(case=case, engines=engines, layers=layers, pos=torch.arange(tokens, device="cuda"),
                 ends=_span_ends(1, tokens))
    for s in range(0, 3 * recent, recent):
        for engine, layer in zip(engines, layers):
            _serve_step(engine, layer, state, s, s + recent)
    return state


# ----------------------------------------------------------------------
# One pass
# ----------------------------------------------------------------------

def _serve_step(engine, layer, state, start, end):
    q, k, v, k_raw = (t[:, :, start:end] for t in layer)
    return engine(q, k, v, k_raw, input_pos=state["pos"][start:end], span_ends=state["ends"][:, start:end])


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("decode", "chunk"):
        with torch.no_grad():
            return log_kv_chunk_attention(state["cache"], state["q"], state["k"], state["v"], case["dim"] ** -0.5,
                                          0.0, reuse_prefix=kind == "decode")
    if kind == "train":
        y = log_kv_chunk_attention(state["cache"], state["q"], state["k"], state["v"], case["dim"] ** -0.5, 0.0)
        return [y.detach(), *torch.autograd.grad(y, (state["q"], state["k"], state["v"]), state["dout"])]
    if kind == "train_stream":
        y = LogKVStreamTrainingAttention.apply(state["q"], state["k"], state["v"], state["cache"],
                                               case["dim"] ** -0.5, case["block"], 0.0, state["k_raw"],
                                               state["ends"])
        return [y.detach(), *torch.autograd.grad(y, (state["q"], state["k"], state["v"]), state["dout"])]
    if kind == "flush":
        cache, n = state["cache"], case["recent"]
        cache.reset_parameters()
        for s in range(0, n * case["blocks"], n):
            ends = state["ends"]
            cache.add_recent(state["k"][:, :, s:s + n], state["v"][:, :, s:s + n],
                             k_raw=state["k_raw"][:, :, s:s + n], input_pos=state["pos"][s:s + n],
                             span_ends=None if ends is None else ends[:, s:s + n])
        names = STATE + (ALPHA_STATE if case["alpha"] else ())
        return {name: getattr(cache, name) for name in names}
    for engine in state["engines"]:
        engine.reset()
    outs, prompt, step = [], case["prompt"], case["recent"]
    for s in range(0, prompt, step):
        outs.append([_serve_step(e, layer, state, s, min(s + step, prompt))
                     for e, layer in zip(state["engines"], state["layers"])])
    for s in range(prompt, prompt + case["decode"]):
        outs.append([_serve_step(e, layer, state, s, s + 1)
                     for e, layer in zip(state["engines"], state["layers"])])
    return [torch.cat(ys, dim=1) for ys in zip(*outs)]


# ----------------------------------------------------------------------
# What a pass cannot do without, and how closely it can be compared
# ----------------------------------------------------------------------

def _prefix_rows(case):
    share = np.full((1, 1, K), _archived(case) // K, dtype=np.int64)
    return int(_slot_counts(case, share).sum()) + (EXACT if case["alpha"] else 0) + case["recent"]


def work(case):
    kind, groups, dim = case["kind"], case["groups"], case["dim"]
    batch = case.get("batch", 1)
    if kind in ("decode", "chunk", "train"):
        rows, prefix, heads = case["rows"], _prefix_rows(case), case["heads"]
        size = torch.empty((), dtype=DTYPES[case["dtype"]]).element_size()
        # Every prefix row's key, mass bias and value once; the queries, current rows and output.
        io = batch * rows * dim * size * (2 * heads + 2 * groups)
        pairs = batch * heads * (rows * prefix + rows * (rows + 1) // 2)
        nbytes = batch * groups * prefix * (2 * dim + 1) * 2 + io
        if kind == "train":   # and the gradients; backward: five products to the forward's two
            return {"bytes": 2 * nbytes + io, "flops": 14 * dim * pairs}
        return {"bytes": nbytes, "flops": 4 * dim * pairs}
    if kind == "flush":
        tokens, recent = case["recent"] * case["blocks"], case["recent"]
        flushed = tokens - recent
        lanes = batch * groups
        from logkv_amd import ladder_budget
        slots, levels, _ = ladder_budget(batch, groups, tokens, dim, dim, B, K, EXACT if case["alpha"] else 0, 2)
        state = lanes * K * levels * slots * (4 * dim + 4 + 4 * 8 + 1) + lanes * 2 * recent * 6 * dim
        flops = lanes * flushed * K * dim * 2
        if case["unified"]:
            flops += lanes * (case["blocks"] - 1) * recent * (recent - 1) // 2 * dim * 3
        return {"bytes": lanes * tokens * dim * 6 + state, "flops": flops}
    # Streams: every token sees at least the window before its block and the block up to it.
    if kind == "train_stream":
        tokens, block, recent, heads, layers, factor = (case["tokens"], case["block"], case["recent"], case["heads"],
                                                        1, 14)
    else:
        tokens, block, recent, heads, layers, factor = (case["prompt"] + case["decode"], case["recent"],
                                                        case["recent"], case["heads"], case["layers"], 4)
    pairs = sum(min(t // block * block, recent) + t % block + 1 for t in range(tokens))
    rows = batch * tokens * dim * 2 * (2 * heads + 3 * groups) * layers
    return {"bytes": rows * (2 if kind == "train_stream" else 1),
            "flops": factor * dim * batch * heads * layers * pairs}


def tolerance(case):
    # A commit's state is decided and rounded in one fixed order: it is the same bit for bit.
    if case["kind"] == "flush":
        return "exact"
    # bf16 outputs of float32 sums over bf16 rows. Against 64 bits, without the roundings of the rotated
    # keys and mass biases to bf16, outputs are 7e-3 off and a chunk's own gradients 2e-3: the same
    # roundings summed in another order differ by about a third of that.
    return {"rel": 1e-2}


# ----------------------------------------------------------------------
# The same outputs in 64 bits
# ----------------------------------------------------------------------

def _prefix64(case, cache_state):
    """Keys, values and log-mass biases of the cache's rows ``[batch, groups, rows, .]``; rows that hold
    nothing have bias -inf."""
    cos, sin = (t.double() for t in _tables(case["context"], case["dim"]))
    batch, groups, dim = case["batch"], case["groups"], case["dim"]
    w = cache_state["level_w"].reshape(batch, groups, -1)
    wi = w.long().clamp(min=1)
    anchor = (2 * cache_state["level_sum_wp"].reshape(batch, groups, -1) + wi) // (2 * wi)
    keys = [_rope(cache_state["level_k"].reshape(batch, groups, -1, dim).double(), cos[anchor], sin[anchor])]
    values = [cache_state["level_v"].reshape(batch, groups, -1, dim).double()]
    biases = [torch.where(w > 0, w.double().clamp(min=1).log(), -math.inf)]
    if case["alpha"]:
        pos, ok = cache_state["alpha_pos"], cache_state["alpha_valid"]
        keys.append(_rope(cache_state["alpha_k_raw"].double(), cos[pos][:, None], sin[pos][:, None]))
        values.append(cache_state["alpha_v"].double())
        biases.append(torch.where(ok, 0.0, -math.inf).double()[:, None].expand(-1, groups, -1))
    keys.append(cache_state["recent_k"].double())
    values.append(cache_state["recent_v"].double())
    biases.append(torch.zeros(batch, groups, case["recent"], dtype=torch.float64, device="cuda"))
    return torch.cat(keys, dim=2), torch.cat(values, dim=2), torch.cat(biases, dim=2)


def exact(case, seed):
    if case["kind"] not in ("decode", "chunk", "train"):
        return None   # decided step by step from earlier results: no value apart from them
    state, rows = _readout_state(case, seed)
    keys, values, bias = _prefix64(case, state)
    q, k, v, dout = (rows[n].double() for n in ("q", "k", "v", "dout"))
    if case["kind"] == "train":
        for t in (q, k, v):
            t.requires_grad_(True)
    n, per = case["rows"], case["heads"] // case["groups"]
    mask = torch.full((n, n), -math.inf, dtype=torch.float64, device="cuda").triu(1)
    scale = case["dim"] ** -0.5
    grads = [torch.zeros_like(t) for t in (q, k, v)]
    out = torch.empty_like(q)
    for b in range(case["batch"]):
        for h in range(case["heads"]):
            grp = h // per
            kk, vv = torch.cat((keys[b, grp], k[b, grp])), torch.cat((values[b, grp], v[b, grp]))
            logits = scale * (q[b, h] @ kk.T)
            extra = torch.cat((bias[b, grp][None].expand(n, -1), mask), dim=1)
            y = torch.softmax(logits + extra, dim=-1) @ vv
            if case["kind"] == "train":
                for into, t in zip(grads, torch.autograd.grad(y, (q, k, v), dout[b, h])):
                    into += t
            out[b, h] = y.detach()
    return [out, *grads] if case["kind"] == "train" else out
