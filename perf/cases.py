"""The attention and gated-delta work that a serving program has this library do, as measurable cases.

Every case is the Qwen3.5 layer shape that the library and its benchmark use: 16 query / 4 KV heads of 256
dims for the gated attention, 16 key / 32 value heads of 128 dims for the gated delta rule.  Calls go through
raftinfer_amd.ops, with the KV caches, workspaces and states that a serving program owns.  A token step
(kinds "decode" and "delta_decode") is replayed from a HIP graph of all layers of the kind, as the executor
replays its decode step; prompts and the batched decode are enqueued call by call.

    import perf.cases as c
    state = c.prepare(c.listed()[0], seed=1)
    outputs = c.run(state)
"""
from __future__ import annotations

import math

import numpy as np
import torch

from raftinfer_amd import ops

HQ, HKV, D = 16, 4, 256          # attention: query heads, KV heads, head dim
HK, HV, DK = 16, 32, 128         # gated delta: key heads, value heads, key and value dim
HIDDEN = HV * DK
CONV_DIM = 2 * HK * DK + HV * DK
ROW = CONV_DIM + 2 * HV + HIDDEN  # packed delta row: q k v | beta | alpha | gate
CONV_W, EPS = 4, 1e-6
ROTARY, ROPE_BASE = 64, 1e7
WIDE = torch.float64

_stream = None


def stream():
    """The one stream that the program enqueues everything on (the library takes no null stream)."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
        torch.cuda.set_stream(_stream)
    return _stream


# ------------------------------------------------------------------ cases

def listed():
    return [
        # One token of a short chat, 8 attention layers replayed from a graph: latency and launches.
        {"name": "decode_short", "kind": "decode", "layers": 8, "context": 201, "max_context": 4096, "f32_cache": False},
        # One token at the benchmark's headline context (bf16 head-major cache, 256-token partitions).
        {"name": "decode_4096", "kind": "decode", "layers": 8, "context": 4096, "max_context": 4096, "f32_cache": False},
        # One token of a long document, ragged end.
        {"name": "decode_long", "kind": "decode", "layers": 2, "context": 60001, "max_context": 65536, "f32_cache": False},
        # The execution policy's default cache: f32, token-major.
        {"name": "decode_f32_cache", "kind": "decode", "layers": 8, "context": 3000, "max_context": 4096, "f32_cache": True},
        # A serving batch of 32 sequences of very different lengths (the benchmark's batched decode).
        {"name": "decode_batched", "kind": "batched", "sequences": 32, "max_context": 32768, "lengths_seed": 4},
        # The executor's prompt bucket of 512 tokens, start of a prompt (the benchmark's PP512).
        {"name": "prefill_512", "kind": "prefill", "tokens": 512, "past": 0, "max_context": 4096, "f32_cache": False, "fused": False},
        # A later 512-token chunk of a longer prompt, q / k producers fused into the call.
        {"name": "prefill_chunk", "kind": "prefill", "tokens": 512, "past": 3584, "max_context": 4096, "f32_cache": False, "fused": True},
        # A long prompt in one call, ragged end.
        {"name": "prefill_long", "kind": "prefill", "tokens": 6001, "past": 0, "max_context": 8192, "f32_cache": False, "fused": False},
        # The prompt bucket on the execution policy's default cache: f32, token-major.
        {"name": "prefill_f32_cache", "kind": "prefill", "tokens": 512, "past": 0, "max_context": 4096, "f32_cache": True, "fused": False},
        # One token through 24 delta layers, replayed from a graph.
        {"name": "delta_decode", "kind": "delta_decode", "layers": 24, "unpacked": False},
        # The executor's prompt bucket through one delta layer (the benchmark's T = 512).
        {"name": "delta_prefill_512", "kind": "delta_prefill", "tokens": 512, "unpacked": False},
        # A long prompt through one delta layer, ragged end, projections read in place.
        {"name": "delta_prefill_long", "kind": "delta_prefill", "tokens": 4001, "unpacked": True},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "batched", "prefill", "prefill", "prefill", "delta_decode", "delta_prefill", "delta_prefill"])
    if kind == "decode":
        context = _log_int(rng, 1, 65536)
        f32 = rng.random() < 0.3
        most = max(1, min(8, 131072 // (context * (2 if f32 else 1))))
        return {"kind": kind, "layers": rng.randint(1, most), "context": context,
                "max_context": min(65536, 1 << max(12, (context - 1).bit_length())), "f32_cache": f32}
    if kind == "batched":
        return {"kind": kind, "sequences": _log_int(rng, 2, 32), "max_context": _log_int(rng, 300, 32768),
                "lengths_seed": rng.randrange(1 << 16)}
    if kind == "prefill":
        if rng.random() < 0.25:  # the default policy's cache: prompts and chunks of up to 512 tokens
            tokens, past = _log_int(rng, 2, 512), rng.choice([0, rng.randint(1, 512)])
            return {"kind": kind, "tokens": tokens, "past": past, "max_context": 4096, "f32_cache": True, "fused": False}
        if rng.random() < 0.5:   # a chunk of the executor's size or less behind a past
            tokens, past = _log_int(rng, 2, 512), _log_int(rng, 1, 32000)
        else:                    # a whole prompt
            tokens, past = _log_int(rng, 2, 6001), 0
        return {"kind": kind, "tokens": tokens, "past": past, "max_context": 1 << max(12, (tokens + past - 1).bit_length()),
                "f32_cache": False, "fused": rng.random() < 0.4}
    if kind == "delta_decode":
        return {"kind": kind, "layers": rng.randint(1, 24), "unpacked": rng.random() < 0.4}
    return {"kind": kind, "tokens": _log_int(rng, 2, 4001), "unpacked": rng.random() < 0.4}


# ------------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape, dtype=torch.bfloat16):
    return torch.randn(*shape, generator=g, device="cuda", dtype=dtype)


def _lengths(case):
    r = np.random.default_rng(case["lengths_seed"])
    return [int(x) for x in r.integers(1, case["max_context"] + 1, size=case["sequences"])]


def _heavy_keys(g, keys):
    """About 1% of the key rows eight times as large, so that the softmax has maxima to find."""
    rows = torch.rand(keys.shape[:-1], generator=g, device="cuda") < 0.01
    keys[rows] *= 8


def _captured(calls, keep):
    """A HIP graph of `calls`, after one eager pass; the tensors of `keep` hold their values again afterwards."""
    s = stream()
    saved = [t.clone() for t in keep]
    calls()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        calls()
    torch.cuda.set_stream(s)
    for t, old in zip(keep, saved):
        t.copy_(old)
    return graph


def _prepare_decode(case, seed):
    g, s = _gen(seed), stream()
    n, ctx, mx, f32 = case["layers"], case["context"], case["max_context"], case["f32_cache"]
    st = {"kind": "decode"}
    # f32 caches are token-major [2][max][4][256], bf16 caches head-major [2][4][max][256]; rows past the
    # context are never read
    if f32:
        cache = torch.zeros(n, 2, mx, HKV, D, device="cuda", dtype=torch.float32)
        cache[:, :, :ctx] = _randn(g, n, 2, ctx, HKV, D, dtype=torch.float32).bfloat16().float()
        _heavy_keys(g, cache[:, 0, :ctx])
        cache[:, :, ctx - 1] = 0
    else:
        cache = torch.zeros(n, 2, HKV, mx, D, device="cuda", dtype=torch.bfloat16)
        cache[..., :ctx, :] = _randn(g, n, 2, HKV, ctx, D)
        _heavy_keys(g, cache[:, 0, :, :ctx])
        cache[..., ctx - 1, :] = 0
    st["cache"] = cache
    st["q"], st["gate"] = _randn(g, n, HQ, D), _randn(g, n, HQ, D)
    st["k"], st["v"] = _randn(g, n, HKV, D), _randn(g, n, HKV, D)
    st["out"] = torch.empty(n, HQ, D, device="cuda", dtype=torch.bfloat16)
    shape = ops.Qwen35AttentionShape(1, HQ, HKV, D, mx, 0)
    plan = ops.qwen35_online_decode_plan(shape, ops.AUTO, ctx)
    st["ws"] = torch.empty(max(16, ops.qwen35_online_decode_workspace_layout(shape, plan[0])[4]), device="cuda", dtype=torch.uint8)
    st["position"] = torch.tensor([ctx - 1], device="cuda", dtype=torch.int32)

    def calls():
        for i in range(n):
            ops.qwen35_online_attention_decode(
                st["q"][i], st["k"][i], st["v"][i], st["gate"][i], st["out"][i], cache[i], st["ws"], shape, ops.DTYPE_BF16,
                ops.CACHE_F32 if f32 else ops.CACHE_BF16, ops.TOKEN_MAJOR if f32 else ops.HEAD_MAJOR,
                plan=plan, device_position=st["position"], stream=s)
    st["graph"] = _captured(calls, [])
    return st


def _prepare_batched(case, seed):
    g = _gen(seed)
    stream()
    n, mx = case["sequences"], case["max_context"]
    cache = torch.empty(n, 2, HKV, mx, D, device="cuda", dtype=torch.bfloat16)
    for i in range(n):
        cache[i] = _randn(g, 2, HKV, mx, D)
    stride = 2 * HKV * mx * D * 2
    return {"kind": "batched", "cache": cache, "stride": stride, "max": mx,
            "lengths": torch.tensor(_lengths(case), device="cuda", dtype=torch.int32),
            "q": _randn(g, n, HQ, D), "gate": _randn(g, n, HQ, D), "k": _randn(g, n, HKV, D), "v": _randn(g, n, HKV, D),
            "out": torch.empty(n, HQ, D, device="cuda", dtype=torch.bfloat16),
            "ws": torch.empty(ops.qwen35_batched_decode_workspace_bytes(n, mx, stride), device="cuda", dtype=torch.uint8)}


def _prepare_prefill(case, seed):
    g = _gen(seed)
    stream()
    t, past, mx, f32 = case["tokens"], case["past"], case["max_context"], case["f32_cache"]
    st = {"kind": "prefill", "f32": f32, "fused": case["fused"], "shape": ops.Qwen35AttentionShape(t, HQ, HKV, D, mx, past)}
    if f32:
        st["cache"] = torch.zeros(2, mx, HKV, D, device="cuda", dtype=torch.float32)
        st["cache"][:, :past] = _randn(g, 2, past, HKV, D).float()
    else:
        st["cache"] = torch.zeros(2, HKV, mx, D, device="cuda", dtype=torch.bfloat16)
        st["cache"][:, :, :past] = _randn(g, 2, HKV, past, D)
    st["k"], st["v"] = _randn(g, t, HKV, D), _randn(g, t, HKV, D)
    st["out"] = torch.empty(t, HQ, D, device="cuda", dtype=torch.bfloat16)
    if case["fused"]:
        st["qg"] = _randn(g, t, HQ, 2, D)
        st["norm"] = ops.Qwen35FusedNormRope(1 + 0.1 * _randn(g, D), 1 + 0.1 * _randn(g, D), ROTARY, ROPE_BASE, EPS)
    else:
        st["q"], st["gate"] = _randn(g, t, HQ, D), _randn(g, t, HQ, D)
        st["policy"] = ops.Qwen35AttentionLaunchPolicy(
            ops.ONLINE_TILED, ops.CACHE_F32 if f32 else ops.CACHE_BF16, ops.TOKEN_MAJOR if f32 else ops.HEAD_MAJOR)
    return st


def _delta_weights(g, n):
    return {"conv_w": 0.3 * _randn(g, n, CONV_DIM, CONV_W), "a": -torch.exp(0.5 * _randn(g, n, HV, dtype=torch.float32)).bfloat16(),
            "dt": _randn(g, n, HV), "norm": _randn(g, n, DK)}


def _delta_inputs(g, unpacked, *lead):
    if not unpacked:
        return {"row": _randn(g, *lead, ROW)}
    return {"qkv": _randn(g, *lead, CONV_DIM), "beta": _randn(g, *lead, HV), "alpha": _randn(g, *lead, HV), "z": _randn(g, *lead, HIDDEN)}


def _delta_call(st, shape, i, s):
    w = (st["conv_w"][i], st["a"][i], st["dt"][i], st["norm"][i], st["out"][i], st["conv"][i], st["rec"][i], st["ws"], shape,
         ops.DTYPE_BF16, ops.DTYPE_BF16)
    if "row" in st:
        ops.qwen35_gated_delta(st["row"][i], *w, stream=s)
    else:
        ops.qwen35_gated_delta_unpacked(st["qkv"][i], st["beta"][i], st["alpha"][i], st["z"][i], *w, stream=s)


def _prepare_delta(case, seed):
    g, s = _gen(seed), stream()
    n, t = case.get("layers", 1), case.get("tokens", 1)
    shape = ops.GatedDeltaShape(t, HIDDEN, HK, HV, DK, DK, CONV_W, EPS)
    st = {"kind": case["kind"], "shape": shape, **_delta_weights(g, n), **_delta_inputs(g, case["unpacked"], n, t)}
    st["conv"] = _randn(g, n, CONV_DIM, CONV_W - 1).float()
    st["rec"] = 0.05 * _randn(g, n, HV, DK, DK, dtype=torch.float32)
    st["out"] = torch.empty(n, t, HIDDEN, device="cuda", dtype=torch.bfloat16)
    st["ws"] = torch.empty(ops.qwen35_gated_delta_workspace_bytes(shape), device="cuda", dtype=torch.uint8)
    if case["kind"] == "delta_decode":
        def calls():
            for i in range(n):
                _delta_call(st, shape, i, s)
        st["graph"] = _captured(calls, [st["conv"], st["rec"]])
    return st


def prepare(case, seed):
    make = {"decode": _prepare_decode, "batched": _prepare_batched, "prefill": _prepare_prefill}.get(case["kind"], _prepare_delta)
    return make(case, seed)


# ------------------------------------------------------------------ one pass

def run(st):
    kind = st["kind"]
    if kind == "decode":
        st["graph"].replay()
        return {"out": st["out"], "cache": st["cache"]}
    if kind == "delta_decode":
        st["graph"].replay()
        return {"out": st["out"], "conv": st["conv"], "rec": st["rec"]}
    if kind == "batched":
        ops.qwen35_online_attention_decode_batched(st["q"], st["k"], st["v"], st["gate"], st["out"], st["cache"], st["lengths"],
                                                   st["ws"], st["max"], st["stride"], stream=_stream)
        return {"out": st["out"], "cache": st["cache"]}
    if kind == "prefill":
        if st["fused"]:
            ops.qwen35_online_attention_prefill_fused(st["qg"], st["k"], st["v"], st["out"], st["cache"], st["shape"], st["norm"],
                                                      stream=_stream)
        else:
            ops.qwen35_causal_attention(st["q"], st["k"], st["v"], st["gate"], st["out"], st["cache"], None, st["shape"],
                                        ops.DTYPE_BF16, st["policy"], stream=_stream)
        return {"out": st["out"], "cache": st["cache"]}
    _delta_call(st, st["shape"], 0, _stream)
    return {"out": st["out"], "conv": st["conv"], "rec": st["rec"]}


# ------------------------------------------------------------------ what a pass cannot do without

def work(case):
    kind = case["kind"]
    if kind in ("decode", "batched"):
        lengths = _lengths(case) if kind == "batched" else [case["context"]] * case["layers"]
        eb = 4 if case.get("f32_cache") else 2
        keys = sum(lengths)
        # every K / V row read once; q, gate, the new rows read and out, the appended rows written
        return {"bytes": keys * 2 * HKV * D * eb + len(lengths) * (3 * HQ * D * 2 + 2 * HKV * D * (2 + eb)),
                "flops": keys * HQ * D * 4}
    if kind == "prefill":
        t, past = case["tokens"], case["past"]
        eb = 4 if case["f32_cache"] else 2
        pairs = t * past + t * (t + 1) // 2
        return {"bytes": t * (3 * HQ * D * 2 + 2 * HKV * D * (2 + eb)) + past * 2 * HKV * D * eb, "flops": pairs * HQ * D * 4}
    n, t = case.get("layers", 1), case.get("tokens", 1)
    states = 2 * 4 * (CONV_DIM * (CONV_W - 1) + HV * DK * DK) + 2 * (CONV_DIM * CONV_W + 2 * HV + DK)
    return {"bytes": n * (t * (ROW + HIDDEN) * 2 + states), "flops": n * t * (6 * DK * DK * HV + 2 * CONV_W * CONV_DIM)}


def tolerance(case):
    # Four times what the outputs are off the 64-bit result.  bf16 rounding of the outputs alone is 1.7e-3 of
    # the 2-norm and 3.9e-3 of a value at most.  The prefill on a bf16 cache also rounds its probabilities to
    # bf16: up to 2.3e-3 of the 2-norm, and 4.3e-2 of the root mean square at the first tokens of a long
    # prompt, whose outputs are far larger than the others.  States (f32) and appended rows lie far inside.
    if case["kind"] == "prefill" and not case["f32_cache"]:
        return {"rel": 9e-3, "max": 0.17}
    return {"rel": 7e-3, "max": 0.016}


# ------------------------------------------------------------------ the same in 64 bits

def _attention(q, k, v, gate, past):
    """q, gate [T][16][256], k, v [past + T][4][256], all WIDE: causal softmax attention, sigmoid output gate."""
    t, n = q.shape[0], k.shape[0]
    out = torch.empty_like(q)
    at = torch.arange(n, device="cuda")
    for h in range(HQ):
        kh, vh = k[:, h // (HQ // HKV)], v[:, h // (HQ // HKV)]
        for a in range(0, t, 1024):
            b = min(t, a + 1024)
            e = past + b
            score = q[a:b, h] @ kh[:e].T / math.sqrt(D)
            score.masked_fill_(at[None, :e] > past + torch.arange(a, b, device="cuda")[:, None], -math.inf)
            out[a:b, h] = torch.softmax(score, -1) @ vh[:e]
    return out * torch.sigmoid(gate)


def _norm_rope(x, w, past):
    """x [T][heads][256] WIDE: RMSNorm and NeoX rotation of the first ROTARY dims, as the bf16 that attention reads."""
    x = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.to(WIDE)
    half = ROTARY // 2
    p = torch.arange(half, device="cuda", dtype=WIDE)
    theta = (past + torch.arange(x.shape[0], device="cuda", dtype=WIDE))[:, None] / ROPE_BASE ** (2 * p / ROTARY)
    c, s = theta.cos()[:, None], theta.sin()[:, None]
    a, b = x[..., :half], x[..., half:ROTARY]
    return torch.cat([a * c - b * s, a * s + b * c, x[..., ROTARY:]], -1).bfloat16().to(WIDE)


def _exact_decode(case, seed):
    st = _prepare_decode(case, seed)
    ctx, out = case["context"], []
    for i in range(case["layers"]):
        rows = st["cache"][i] if case["f32_cache"] else st["cache"][i].transpose(1, 2)  # [2][max][4][256]
        k, v = (torch.cat([rows[j, :ctx - 1].to(WIDE), st[x][i:i + 1].to(WIDE)]) for j, x in ((0, "k"), (1, "v")))
        out.append(_attention(st["q"][i:i + 1].to(WIDE), k, v, st["gate"][i:i + 1].to(WIDE), ctx - 1)[0])
    return {"out": torch.stack(out), "cache": None}


def _exact_batched(case, seed):
    st = _prepare_batched(case, seed)
    out = []
    for i, n in enumerate(_lengths(case)):
        rows = st["cache"][i].transpose(1, 2)
        k, v = (torch.cat([rows[j, :n - 1].to(WIDE), st[x][i:i + 1].to(WIDE)]) for j, x in ((0, "k"), (1, "v")))
        out.append(_attention(st["q"][i:i + 1].to(WIDE), k, v, st["gate"][i:i + 1].to(WIDE), n - 1)[0])
    return {"out": torch.stack(out), "cache": None}


def _exact_prefill(case, seed):
    st = _prepare_prefill(case, seed)
    t, past = case["tokens"], case["past"]
    rows = st["cache"] if case["f32_cache"] else st["cache"].transpose(1, 2)
    k, v = st["k"].to(WIDE), st["v"].to(WIDE)
    if case["fused"]:
        q, gate = (st["qg"][:, :, j].to(WIDE) for j in (0, 1))
        q, k = _norm_rope(q, st["norm"].query_norm_weight, past), _norm_rope(k, st["norm"].key_norm_weight, past)
    else:
        q, gate = st["q"].to(WIDE), st["gate"].to(WIDE)
    k, v = torch.cat([rows[0, :past].to(WIDE), k]), torch.cat([rows[1, :past].to(WIDE), v])
    return {"out": _attention(q, k, v, gate, past), "cache": None}


def _exact_delta(case, seed):
    st = _prepare_delta({**case, "kind": "delta_prefill"}, seed)
    n, t = case.get("layers", 1), case.get("tokens", 1)
    row = st["row"] if "row" in st else torch.cat([st["qkv"], st["beta"], st["alpha"], st["z"]], -1)
    row = row.view(n, t, ROW).to(WIDE)
    x = torch.cat([st["conv"].to(WIDE).transpose(1, 2), row[..., :CONV_DIM]], 1)  # [n][3 + T][channels]
    w = st["conv_w"].to(WIDE)
    y = sum(x[:, j:j + t] * w[:, None, :, j] for j in range(CONV_W))
    y = y * torch.sigmoid(y)
    q, k, v = y.split([HK * DK, HK * DK, HV * DK], -1)
    unit = lambda z: z * torch.rsqrt((z * z).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    q, k = (unit(z.reshape(n, t, HK, DK)).repeat(1, 1, HV // HK, 1) for z in (q, k))  # value head h reads key head h % HK
    q, v = q / math.sqrt(DK), v.reshape(n, t, HV, DK)
    b, a, z = row[..., CONV_DIM:].split([HV, HV, HIDDEN], -1)
    beta = torch.sigmoid(b)
    decay = torch.exp(st["a"].to(WIDE)[:, None] * torch.nn.functional.softplus(a + st["dt"].to(WIDE)[:, None]))
    s, raw = st["rec"].to(WIDE), torch.empty(n, t, HV, DK, device="cuda", dtype=WIDE)
    for i in range(t):
        s = s * decay[:, i, :, None, None]
        d = (v[:, i] - (s * k[:, i, :, :, None]).sum(2)) * beta[:, i, :, None]
        s = s + k[:, i, :, :, None] * d[:, :, None, :]
        raw[:, i] = (s * q[:, i, :, :, None]).sum(2)
    out = raw * torch.rsqrt((raw * raw).mean(-1, keepdim=True) + EPS) * st["norm"].to(WIDE)[:, None, None]
    return {"out": out.reshape(n, t, HIDDEN) * (z * torch.sigmoid(z)), "conv": x[:, t:].transpose(1, 2).contiguous(), "rec": s}


def exact(case, seed):
    make = {"decode": _exact_decode, "batched": _exact_batched, "prefill": _exact_prefill}.get(case["kind"], _exact_delta)
    return make(case, seed)
