"""The attention work a Qwen3-TTS engine has this library do, as timed cases.

Four kinds of case, over the sizes an engine serves (16 query heads over 8 KV heads, head_dim 128, bf16, 16-token pages):

  decode   one frame of the talker: 28 decode-attention layer calls in a HIP graph, the way the engine replays a frame,
           with the frame's plan when ``planned``.  ``form``: "plain" (K/V already appended), "append" (this step's K/V
           written by the call) or "append_rope" (q/k normalised and rotated by it too, from the raw qkv projection).
  cp       the code predictor's steps over its 16-slot scratch: 3 layers x 16 steps in a HIP graph.
  prefill  one layer of a prompt prefill, called eagerly on ragged packed sequences.  ``form``: "varlen" (packed K/V),
           "paged" (K/V read from the pool), "append" or "append_rope" (the prompt's K/V written to the pool).
  admit    the fast-admission layers: S sequences of R new tokens after a prefix of P, 28 layers in a HIP graph.
           ``form``: "dense", "append" or "append_rope".
"""
from __future__ import annotations

import math
import os
import sys
from types import SimpleNamespace

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen3-tts-engine_amd"))

import q3attn  # noqa: E402

HQ, HKV, D, PAGE = 16, 8, 128, 16
LAYERS = 28          # talker layers
CP_LAYERS, CP_STEPS = 3, 16
SCALE = D ** -0.5
EPS = 1e-6
DEV = "cuda"
BF = torch.bfloat16


def listed():
    return [
        # One stream speaking: the smallest frame, where the launches and the memory latency are the time.
        {"name": "decode_1row", "kind": "decode", "form": "append_rope", "rows": 1, "lo": 700, "hi": 1100, "pads": 0,
         "planned": True, "seed_ctx": 1},
        # A lightly loaded server: one of the small batch buckets.
        {"name": "decode_16rows", "kind": "decode", "form": "append_rope", "rows": 16, "lo": 100, "hi": 1500, "pads": 2,
         "planned": True, "seed_ctx": 2},
        # A middling batch through the append form, as a caller with its own q/k producers makes it.
        {"name": "decode_64rows", "kind": "decode", "form": "append", "rows": 64, "lo": 64, "hi": 1200, "pads": 5,
         "planned": True, "seed_ctx": 3},
        # The drop-in call for flash_attn_with_kvcache after an index_copy_ append, without a plan.
        {"name": "decode_250rows_plain", "kind": "decode", "form": "plain", "rows": 250, "lo": 200, "hi": 1200,
         "pads": 0, "planned": False, "seed_ctx": 4},
        # The full server of the benchmark: 576 seats, a tenth of them empty, log-uniform contexts.
        {"name": "decode_576rows", "kind": "decode", "form": "append_rope", "rows": 576, "lo": 64, "hi": 1800,
         "pads": 58, "planned": True, "seed_ctx": 5},
        # The code predictor of a small batch and of the full server.
        {"name": "cp_8rows", "kind": "cp", "form": "append_rope", "rows": 8},
        {"name": "cp_512rows", "kind": "cp", "form": "append_rope", "rows": 512},
        # One new prompt arriving alone.
        {"name": "prefill_1x300", "kind": "prefill", "form": "append_rope", "seqs": 1, "lo": 300, "hi": 300,
         "causal": True, "seed_ctx": 6},
        # A burst of 32 prompts, the whole prompt step from the raw projections.
        {"name": "prefill_32", "kind": "prefill", "form": "append_rope", "seqs": 32, "lo": 150, "hi": 400,
         "causal": True, "seed_ctx": 7},
        # Long prompts (a long reference recording and text), through the varlen drop-in on packed K/V.
        {"name": "prefill_16_long", "kind": "prefill", "form": "varlen", "seqs": 16, "lo": 512, "hi": 2048,
         "causal": True, "seed_ctx": 8},
        # The fast-admission shape of the engine: 42 new tokens over a 35-token voice prefix.
        {"name": "admit_8x42", "kind": "admit", "form": "append_rope", "seqs": 8, "new": 42, "prefix": 35},
        # Admission with a long text after a long voice prefix, through the flash_attn_func drop-in.
        {"name": "admit_6x210_prefix170", "kind": "admit", "form": "dense", "seqs": 6, "new": 210, "prefix": 170},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "cp", "prefill", "prefill", "admit"])
    if kind == "decode":
        hi = _log_int(rng, 40, 1800)
        lo = max(1, int(hi * rng.uniform(0.05, 1.0)))
        rows = min(_log_int(rng, 1, 576), max(1, int(280000 / (0.5 * (lo + hi)))))
        return {"kind": kind, "form": rng.choice(["plain", "append", "append_rope"]), "rows": rows, "lo": lo, "hi": hi,
                "pads": rng.randrange(0, rows // 8 + 1), "planned": rng.random() < 0.7,
                "seed_ctx": rng.randrange(1 << 20)}
    if kind == "cp":
        return {"kind": kind, "form": rng.choice(["plain", "append", "append_rope"]), "rows": _log_int(rng, 1, 704)}
    if kind == "prefill":
        hi = _log_int(rng, 24, 2048)
        lo = max(1, int(hi * rng.uniform(0.1, 1.0)))
        seqs = min(_log_int(rng, 1, 64), max(1, int(24000 / (0.5 * (lo + hi)))))
        return {"kind": kind, "form": rng.choice(["varlen", "paged", "append", "append_rope", "append_rope"]),
                "seqs": seqs, "lo": lo, "hi": hi, "causal": rng.random() < 0.9, "seed_ctx": rng.randrange(1 << 20)}
    new = _log_int(rng, 4, 320)
    return {"kind": kind, "form": rng.choice(["dense", "append", "append_rope"]), "seqs": rng.randint(1, 8), "new": new,
            "prefix": rng.randrange(0, 200)}


# ---------------------------------------------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _unit(shape, g):
    """Rows of unit RMS (a normalised and rotated q or k: the rotation keeps the norm)."""
    x = torch.randn(shape, generator=g, device=DEV)
    return (x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS)).to(BF)


def _randn(shape, g):
    return torch.randn(shape, generator=g, device=DEV).to(BF)


def _norm_w(g):
    return (0.5 + torch.rand(D, generator=g, device=DEV)).to(BF)


def _rope_rows(pos):
    inv = 1.0e6 ** (-torch.arange(0, D, 2, dtype=torch.float64, device=DEV) / D)
    a = pos.to(DEV).double()[:, None] * inv[None, :]
    a = torch.cat([a, a], dim=-1)
    return a.cos().to(BF), a.sin().to(BF)


def _contexts(case):
    """Context lengths (tokens attended, this step's included), the padded rows (0) at the tail.  They belong to the
    case, not to the seed of the values, so that every pass of a case does the same work."""
    rng = np.random.default_rng(case["seed_ctx"])
    live = case["rows"] - case["pads"]
    lo, hi = case["lo"], case["hi"]
    c = np.rint(np.exp(rng.uniform(math.log(lo), math.log(hi), size=live))) if hi > 4 * lo else rng.integers(lo, hi + 1, live)
    return np.concatenate([c.astype(np.int64), np.zeros(case["pads"], np.int64)])


def _lengths(case):
    rng = np.random.default_rng(case["seed_ctx"])
    return rng.integers(case["lo"], case["hi"] + 1, case["seqs"]).astype(np.int64)


def _pool(pages, g):
    """A K/V pool of earlier tokens, filled in pieces."""
    kc = torch.empty((pages, PAGE, HKV, D), dtype=BF, device=DEV)
    vc = torch.empty_like(kc)
    for c0 in range(0, pages, 8192):
        n = min(8192, pages - c0)
        kc[c0:c0 + n] = _unit((n, PAGE, HKV, D), g)
        vc[c0:c0 + n] = _randn((n, PAGE, HKV, D), g)
    return kc, vc


def _capture(fn):
    """fn's calls in a HIP graph, after one eager pass on a side stream."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


def _decode_inputs(case, seed):
    ctx = _contexts(case)
    B = case["rows"]
    g, rng = _gen(seed), np.random.default_rng(seed)
    used = -(-ctx // PAGE)
    cap = 256 * -(-int(ctx.max() + 1) // 256)        # a seat holds a multiple of 256 positions
    shared = max(16384, 3 * int(used.sum()))
    # The layers share one pool's pages (each through a random table of its own) except each row's last page, which
    # the append forms write: that one belongs to one layer alone.  Entries past a row's pages are unallocated (-1).
    tables = np.full((LAYERS, B, cap // PAGE), -1, np.int32)
    for layer in range(LAYERS):
        ids = rng.permutation(shared)
        at = 0
        for b in range(B):
            n = int(used[b])
            if n:
                tables[layer, b, :n - 1] = ids[at:at + n - 1]
                tables[layer, b, n - 1] = shared + layer * B + b
                at += n - 1
    s = SimpleNamespace(case=case, ctx=ctx, tables_host=tables)
    s.kc, s.vc = _pool(shared + LAYERS * B, g)
    s.tables = torch.from_numpy(tables).to(DEV)
    s.seqlens = torch.from_numpy(ctx if case["form"] == "plain" else ctx - 1).to(torch.int32).to(DEV)
    if case["form"] == "append_rope":
        s.qkv = [_randn((B, (HQ + 2 * HKV) * D), g) for _ in range(LAYERS)]
        s.qn, s.kn = [_norm_w(g) for _ in range(LAYERS)], [_norm_w(g) for _ in range(LAYERS)]
        s.cos, s.sin = _rope_rows(torch.from_numpy(np.maximum(ctx - 1, 0)))
    else:
        s.q = [_unit((B, HQ, D), g) for _ in range(LAYERS)]
        if case["form"] == "append":
            s.k = [_unit((B, HKV, D), g) for _ in range(LAYERS)]
            s.v = [_randn((B, HKV, D), g) for _ in range(LAYERS)]
    return s


def _split_qkv(x):
    n = x.shape[0]
    return (x[:, :HQ * D].view(n, HQ, D), x[:, HQ * D:(HQ + HKV) * D].view(n, HKV, D), x[:, (HQ + HKV) * D:].view(n, HKV, D))


def _decode_frame(s):
    form = s.case["form"]
    plans = q3attn.decode_plan(s.seqlens, s.tables, PAGE, form=form) if s.case["planned"] else None
    outs = []
    for i in range(LAYERS):
        bt, plan = s.tables[i], (plans[i] if plans is not None else None)
        if form == "plain":
            o = q3attn.flash_attn_with_kvcache(s.q[i].unsqueeze(1), s.kc, s.vc, cache_seqlens=s.seqlens, block_table=bt,
                                               softmax_scale=SCALE, causal=True, scheduler_metadata=plan)
        elif form == "append":
            o = q3attn.flash_attn_with_kvcache(s.q[i].unsqueeze(1), s.kc, s.vc, k=s.k[i].unsqueeze(1),
                                               v=s.v[i].unsqueeze(1), cache_seqlens=s.seqlens, block_table=bt,
                                               softmax_scale=SCALE, causal=True, scheduler_metadata=plan)
        else:
            q, k, v = _split_qkv(s.qkv[i])
            o = q3attn.paged_decode_append_rope(q, k, v, s.qn[i], s.kn[i], s.cos, s.sin, s.kc, s.vc, s.seqlens, bt,
                                                SCALE, EPS, plan=plan)
        outs.append(o)
    return outs


def _cp_inputs(case, seed):
    g, B = _gen(seed), case["rows"]
    s = SimpleNamespace(case=case)
    shape = (CP_LAYERS, B, HKV, CP_STEPS, D)
    s.K, s.V = (_unit(shape, g), _randn(shape, g)) if case["form"] == "plain" else \
        (torch.zeros(shape, dtype=BF, device=DEV), torch.zeros(shape, dtype=BF, device=DEV))
    if case["form"] == "append_rope":
        s.qkv = [[_randn((B, (HQ + 2 * HKV) * D), g) for _ in range(CP_LAYERS)] for _ in range(CP_STEPS)]
        s.qn, s.kn = [_norm_w(g) for _ in range(CP_LAYERS)], [_norm_w(g) for _ in range(CP_LAYERS)]
        s.cos, s.sin = _rope_rows(torch.arange(CP_STEPS))
    else:
        s.q = [[_unit((B, HQ, D), g) for _ in range(CP_LAYERS)] for _ in range(CP_STEPS)]
        if case["form"] == "append":
            s.k = [[_unit((B, HKV, D), g) for _ in range(CP_LAYERS)] for _ in range(CP_STEPS)]
            s.v = [[_randn((B, HKV, D), g) for _ in range(CP_LAYERS)] for _ in range(CP_STEPS)]
    return s


def _cp_frame(s):
    outs, form = [], s.case["form"]
    for p in range(CP_STEPS):
        for i in range(CP_LAYERS):
            if form == "plain":
                o = q3attn.cp_attn(s.q[p][i], s.K[i], s.V[i], p + 1, SCALE)
            elif form == "append":
                o = q3attn.cp_attn_append(s.q[p][i], s.k[p][i], s.v[p][i], s.K[i], s.V[i], p, SCALE)
            else:
                q, k, v = _split_qkv(s.qkv[p][i])
                o = q3attn.cp_attn_append_rope(q, k, v, s.K[i], s.V[i], p, SCALE, s.qn[i], s.kn[i], s.cos[p], s.sin[p],
                                               EPS)
            outs.append(o)
    return outs


def _prefill_inputs(case, seed):
    lens = _lengths(case)
    g, rng = _gen(seed), np.random.default_rng(seed)
    T, n = int(lens.sum()), len(lens)
    s = SimpleNamespace(case=case, lens=lens, max_len=int(lens.max()))
    s.cu = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)).to(DEV)
    qkv = _randn((T, (HQ + 2 * HKV) * D), g)
    s.q, s.k, s.v = _split_qkv(qkv)                   # v stays a view of the projection in every form
    if case["form"] == "append_rope":
        s.qn, s.kn = _norm_w(g), _norm_w(g)
        s.cos, s.sin = _rope_rows(torch.from_numpy(np.concatenate([np.arange(x) for x in lens])))
    else:
        s.q, s.k = _unit((T, HQ, D), g), _unit((T, HKV, D), g)
    if case["form"] != "varlen":
        used = -(-lens // PAGE)
        width = int(used.max())
        pages = int(used.sum()) + 64
        ids, table, at = rng.permutation(pages), np.full((n, width), -1, np.int32), 0
        for b in range(n):
            table[b, :used[b]] = ids[at:at + used[b]]
            at += int(used[b])
        s.table = torch.from_numpy(table).to(DEV)
        s.slots = torch.from_numpy(np.concatenate(
            [table[b, np.arange(x) // PAGE].astype(np.int64) * PAGE + np.arange(x) % PAGE for b, x in enumerate(lens)])).to(DEV)
        s.kc = torch.zeros((pages, PAGE, HKV, D), dtype=BF, device=DEV)
        s.vc = torch.zeros_like(s.kc)
        if case["form"] == "paged":
            s.kc.view(-1, HKV, D).index_copy_(0, s.slots, s.k)
            s.vc.view(-1, HKV, D).index_copy_(0, s.slots, s.v)
    return s


def _admit_inputs(case, seed):
    g, rng = _gen(seed), np.random.default_rng(seed)
    S, R, P = case["seqs"], case["new"], case["prefix"]
    n = P + R
    s = SimpleNamespace(case=case)
    if case["form"] == "append_rope":
        s.qkv = [_randn((S, R, (HQ + 2 * HKV) * D), g) for _ in range(LAYERS)]
        s.voices = 4
        s.pk = [_unit((s.voices, P, HKV, D), g) for _ in range(LAYERS)]
        s.pv = [_randn((s.voices, P, HKV, D), g) for _ in range(LAYERS)]
        s.voice = torch.from_numpy(rng.integers(0, s.voices, S)).to(DEV)
        s.qn, s.kn = [_norm_w(g) for _ in range(LAYERS)], [_norm_w(g) for _ in range(LAYERS)]
        s.cos, s.sin = _rope_rows(torch.arange(P, n))
    else:
        s.q = [_unit((S, R, HQ, D), g) for _ in range(LAYERS)]
        s.k = [_unit((S, n, HKV, D), g) for _ in range(LAYERS)]
        s.v = [_randn((S, n, HKV, D), g) for _ in range(LAYERS)]
    if case["form"] != "dense":
        w = -(-n // PAGE)
        s.table = torch.from_numpy(rng.permutation(S * w).reshape(S, w).astype(np.int32)).to(DEV)
        s.kc = torch.zeros((LAYERS, S * w, PAGE, HKV, D), dtype=BF, device=DEV)
        s.vc = torch.zeros_like(s.kc)
    return s


def _admit_layers(s):
    outs, c = [], s.case
    for i in range(LAYERS):
        if c["form"] == "dense":
            o = q3attn.flash_attn_func(s.q[i], s.k[i], s.v[i], softmax_scale=SCALE, causal=True)
        elif c["form"] == "append":
            o = q3attn.prefill_dense_append(s.q[i], s.k[i], s.v[i], s.kc[i], s.vc[i], s.table, SCALE, True)
        else:
            S, R = c["seqs"], c["new"]
            q, k, v = (x.view(S, R, -1, D) for x in torch.split(s.qkv[i], [HQ * D, HKV * D, HKV * D], dim=2))
            o = q3attn.prefill_dense_append_rope(q, k, v, s.pk[i], s.pv[i], s.qn[i], s.kn[i], s.cos, s.sin, s.kc[i],
                                                 s.vc[i], s.table, SCALE, s.voice, True, EPS)
        outs.append(o)
    return outs


def _inputs(case, seed):
    return {"decode": _decode_inputs, "cp": _cp_inputs, "prefill": _prefill_inputs, "admit": _admit_inputs}[
        case["kind"]](case, seed)


def prepare(case, seed):
    s = _inputs(case, seed)
    body = {"decode": _decode_frame, "cp": _cp_frame, "admit": _admit_layers}.get(case["kind"])
    if body is not None:
        s.graph, s.outs = _capture(lambda: body(s))
    return s


# ---------------------------------------------------------------------------------------------------- a pass

def run(s):
    case = s.case
    form = case["form"]
    if case["kind"] == "prefill":
        if form == "varlen":
            return q3attn.flash_attn_varlen_func(s.q, s.k, s.v, s.cu, s.cu, s.max_len, s.max_len, softmax_scale=SCALE,
                                                 causal=case["causal"])
        if form == "paged":
            return q3attn.flash_attn_varlen_func(s.q, s.kc, s.vc, s.cu, s.cu, s.max_len, s.max_len, softmax_scale=SCALE,
                                                 causal=case["causal"], block_table=s.table)
        if form == "append":
            o = q3attn.prefill_append(s.q, s.k, s.v, s.cu, s.cu, s.max_len, s.kc, s.vc, s.table, SCALE, case["causal"])
        else:
            o = q3attn.prefill_append_rope(s.q, s.k, s.v, s.qn, s.kn, s.cos, s.sin, s.cu, s.max_len, s.kc, s.vc, s.table,
                                           SCALE, case["causal"], EPS)
        return {"out": o, "k_cache": s.kc, "v_cache": s.vc}
    s.graph.replay()
    if case["kind"] == "cp":
        return {"out": s.outs} if form == "plain" else {"out": s.outs, "K": s.K, "V": s.V}
    if form in ("plain", "dense"):
        return {"out": s.outs}
    return {"out": s.outs, "k_cache": s.kc, "v_cache": s.vc}


def work(case):
    row_q, row_kv = HQ * D, 2 * HKV * D               # elements of a token's q (or o) and of its K and V
    form = case["form"]
    if case["kind"] == "decode":
        ctx = _contexts(case)
        tok, B, live = int(ctx.sum()), case["rows"], case["rows"] - case["pads"]
        el = tok * row_kv + 2 * B * row_q
        if form != "plain":
            el += live * row_kv                       # the new rows are read from their own tensors and written too
        by = 2 * el + 4 * int((-(-ctx // PAGE)).sum()) + 4 * B
        if form == "append_rope":
            by += 2 * (2 * B * D + 2 * D)
        return {"bytes": LAYERS * by, "flops": LAYERS * 4 * HQ * D * tok}
    if case["kind"] == "cp":
        B = case["rows"]
        el = sum(B * ((p + 1) * row_kv + 2 * row_q + (row_kv if form != "plain" else 0)) for p in range(CP_STEPS))
        return {"bytes": CP_LAYERS * 2 * el, "flops": CP_LAYERS * 4 * HQ * D * B * sum(range(1, CP_STEPS + 1))}
    if case["kind"] == "prefill":
        lens = _lengths(case)
        T = int(lens.sum())
        el = T * (2 * row_q + row_kv * (2 if form.startswith("append") else 1) + (2 * D if form == "append_rope" else 0))
        seen = int((lens * (lens + 1) // 2).sum()) if case["causal"] else int((lens * lens).sum())
        return {"bytes": 2 * el, "flops": 4 * HQ * D * seen}
    S, R, P = case["seqs"], case["new"], case["prefix"]
    el = S * (2 * R * row_q + (P + R) * row_kv * (2 if form != "dense" else 1)) + (2 * R * D if form == "append_rope" else 0)
    return {"bytes": LAYERS * 2 * el, "flops": LAYERS * 4 * HQ * D * S * (R * P + R * (R + 1) // 2)}


def tolerance(case):
    """bf16 inputs and outputs with float32 sums: an output is within half a bf16 step (2^-9) of its value, and P (and
    for the raw forms q and k) carries a rounding of the same size.  Measured against float64: 1.7e-3 to 3.5e-3."""
    return {"rel": 1e-2}


# ------------------------------------------------------------------------------------------ the same in 64 bits

def _x_norm_rope(x, w, cos, sin):
    x, w, cos, sin = x.double(), w.double(), cos.double(), sin.double()
    y = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w
    return y * cos + torch.cat((-y[..., D // 2:], y[..., :D // 2]), dim=-1) * sin


def _x_attend(q, k, v, visible=None):
    """q [N, 16, D] over k, v [L, 8, D] in float64 -> [N, 16, D]; visible [N, L]."""
    n, length = q.shape[0], k.shape[0]
    if length == 0:
        return torch.zeros((n, HQ, D), dtype=torch.float64, device=DEV)
    qh = q.double().view(n, HKV, HQ // HKV, D).permute(1, 2, 0, 3).reshape(HKV, -1, D)
    a = (qh @ k.double().permute(1, 2, 0).contiguous()) * SCALE
    if visible is not None:
        a = a.view(HKV, HQ // HKV, n, length).masked_fill(~visible, -math.inf).view(HKV, -1, length)
    o = torch.softmax(a, dim=-1) @ v.double().permute(1, 0, 2).contiguous()
    return o.view(HKV, HQ // HKV, n, D).permute(2, 0, 1, 3).reshape(n, HQ, D)


def _x_decode(s):
    case, ctx = s.case, s.ctx
    form = case["form"]
    kc, vc = s.kc, s.vc
    if form != "plain":
        kc, vc = kc.double(), vc.double()
    outs = []
    for i in range(LAYERS):
        if form == "append_rope":
            q, k, v = _split_qkv(s.qkv[i])
            q = _x_norm_rope(q, s.qn[i], s.cos[:, None], s.sin[:, None])
            k = _x_norm_rope(k, s.kn[i], s.cos[:, None], s.sin[:, None])
        else:
            q = s.q[i]
            k, v = (s.k[i], s.v[i]) if form == "append" else (None, None)
        o = torch.zeros((case["rows"], HQ, D), dtype=torch.float64, device=DEV)
        for b in range(case["rows"]):
            c = int(ctx[b])
            if c == 0:
                continue
            n = -(-c // PAGE)
            if form != "plain":
                page = int(s.tables_host[i, b, n - 1])
                kc[page, (c - 1) % PAGE] = k[b].double()
                vc[page, (c - 1) % PAGE] = v[b].double()
            pages = s.tables[i, b, :n].long()
            o[b] = _x_attend(q[b:b + 1], kc[pages].view(-1, HKV, D)[:c], vc[pages].view(-1, HKV, D)[:c])[0]
        outs.append(o if form == "append_rope" else o.unsqueeze(1))
    return {"out": outs} if form == "plain" else {"out": outs, "k_cache": kc, "v_cache": vc}


def _x_cp(s):
    form, B = s.case["form"], s.case["rows"]
    K, V = s.K.double(), s.V.double()
    outs = []
    for p in range(CP_STEPS):
        for i in range(CP_LAYERS):
            if form == "append_rope":
                q, k, v = _split_qkv(s.qkv[p][i])
                q, k = (_x_norm_rope(x, w, s.cos[p], s.sin[p]) for x, w in ((q, s.qn[i]), (k, s.kn[i])))
            else:
                q = s.q[p][i]
                k, v = (s.k[p][i], s.v[p][i]) if form == "append" else (None, None)
            if k is not None:
                K[i, :, :, p], V[i, :, :, p] = k.double(), v.double()
            a = q.double().view(B, HKV, HQ // HKV, D) @ K[i, :, :, :p + 1].transpose(-1, -2).contiguous() * SCALE
            outs.append((torch.softmax(a, dim=-1) @ V[i, :, :, :p + 1].contiguous()).reshape(B, HQ * D))
    return {"out": outs} if form == "plain" else {"out": outs, "K": K, "V": V}


def _x_prefill(s):
    form, causal = s.case["form"], s.case["causal"]
    q, k, v = s.q, s.k, s.v
    if form == "append_rope":
        q = _x_norm_rope(q, s.qn, s.cos[:, None], s.sin[:, None])
        k = _x_norm_rope(k, s.kn, s.cos[:, None], s.sin[:, None])
    out, t0 = torch.empty((q.shape[0], HQ, D), dtype=torch.float64, device=DEV), 0
    for n in (int(x) for x in s.lens):
        at = torch.arange(n, device=DEV)
        out[t0:t0 + n] = _x_attend(q[t0:t0 + n], k[t0:t0 + n], v[t0:t0 + n], at[None, :] <= at[:, None] if causal else None)
        t0 += n
    if not form.startswith("append"):
        return out
    kc, vc = s.kc.double(), s.vc.double()
    kc.view(-1, HKV, D).index_copy_(0, s.slots, k.double())
    vc.view(-1, HKV, D).index_copy_(0, s.slots, v.double())
    return {"out": out, "k_cache": kc, "v_cache": vc}


def _x_admit(s):
    c = s.case
    S, R, P = c["seqs"], c["new"], c["prefix"]
    n = P + R
    seen = torch.arange(n, device=DEV)[None, :] <= P + torch.arange(R, device=DEV)[:, None]
    outs = []
    if c["form"] != "dense":
        kc, vc = s.kc.double(), s.vc.double()
        table = s.table.long()
    for i in range(LAYERS):
        if c["form"] == "append_rope":
            q, k, v = (x.view(S, R, -1, D) for x in torch.split(s.qkv[i], [HQ * D, HKV * D, HKV * D], dim=2))
            q = _x_norm_rope(q, s.qn[i], s.cos[:, None], s.sin[:, None])
            k = torch.cat((s.pk[i][s.voice].double(), _x_norm_rope(k, s.kn[i], s.cos[:, None], s.sin[:, None])), dim=1)
            v = torch.cat((s.pv[i][s.voice], v), dim=1).double()
        else:
            q, k, v = s.q[i], s.k[i].double(), s.v[i].double()
        outs.append(torch.stack([_x_attend(q[j], k[j], v[j], seen) for j in range(S)]))
        if c["form"] != "dense":
            pos = torch.arange(n, device=DEV)
            slots = (table[:, pos // PAGE] * PAGE + pos % PAGE).reshape(-1)
            kc[i].view(-1, HKV, D).index_copy_(0, slots, k.reshape(-1, HKV, D))
            vc[i].view(-1, HKV, D).index_copy_(0, slots, v.reshape(-1, HKV, D))
    return {"out": outs} if c["form"] == "dense" else {"out": outs, "k_cache": kc, "v_cache": vc}


def exact(case, seed):
    s = _inputs(case, seed)
    return {"decode": _x_decode, "cp": _x_cp, "prefill": _x_prefill, "admit": _x_admit}[case["kind"]](s)
