"""The work a serving program has this package do, as measurable cases.

A speculative-decoding engine calls the ops of `ninfer_amd.ops` on device memory of its own: verify
attention over a KV cache (one sequence or a ragged batch, chains and draft trees, the three head
geometries, INT8-G64 and BF16 caches), prompt attention through the same entry points, the
recurrent-state ops of the hybrid layers (verify rounds and prompts), the Q6 output head, the
acceptance samplers and the cache commit, and whole rounds captured once in a graph and replayed.
Every case passes through those entry points on torch-owned memory. Sizes come from the package's
benchmark and tests or are generic.
"""
from __future__ import annotations

import math
import random

import torch

import ninfer_amd as na
from ninfer_amd import ops
from ninfer_amd.device import DeviceBuffer, Graph, Stream

VOCAB = 248320
DEV = "cuda"
# (query heads, KV heads, head_dim): the verify geometry and the two registered head_dim-256 ones
GEOMETRIES = ((40, 8, 128), (24, 4, 256), (16, 2, 256))


# ---- the cases -------------------------------------------------------------------------------

def _attn(**kw):
    c = dict(kind="attention", q_heads=40, kv_heads=8, head_dim=128, cache="int8", tokens=4, batch=1, context=7680,
             context_min=0, tree=False, outliers=False, out="bf16")
    c.update(kw)
    return c


def _hybrid(**kw):
    c = dict(kind="hybrid", head_dim=128, qk_heads=16, value_heads=48, tokens=4, layers=1, snapshot=True)
    c.update(kw)
    return c


def _head(**kw):
    c = dict(kind="head", hidden=5120, drafts=3, batch=1, fused=False, temperature=0.0)
    c.update(kw)
    return c


def listed():
    return [
        # one plain decode step of a short chat, called eagerly: launches and host latency
        _attn(name="decode_short", tokens=1, context=517),
        # the whole greedy verify round of an engine, one captured graph: prepare, 16 attention
        # layers, output head, argmax, accept, hidden-row selection, alignment ids, state slot
        dict(name="round_7k", kind="round", layers=16, context=7680, drafts=3, hidden=5120),
        # one verify layer at the longest context, keys and values with outliers
        _attn(name="verify_260k", context=260096, outliers=True),
        # a ragged batch of 16 sequences, then the rollback of its rejected rows
        _attn(name="verify_batch16", batch=16, context=32768, context_min=1024),
        # 8 draft trees of 16 nodes: tree attention, path acceptance, path compaction
        _attn(name="verify_tree8", batch=8, tokens=16, context=131072, context_min=1024, tree=True),
        # five drafts at a registered head_dim-256 geometry over a BF16 cache
        _attn(name="verify_d256_bf16", q_heads=24, kv_heads=4, head_dim=256, cache="bf16", tokens=6, context=32768),
        # a prompt chunk appended to a running conversation
        _attn(name="prompt_2k", tokens=2048, context=2048),
        # a first prompt of an odd length at a registered head_dim-256 geometry
        _attn(name="prompt_d256", q_heads=24, kv_heads=4, head_dim=256, tokens=1000, context=0),
        # one hybrid layer over a prompt: convolution and recurrence
        _hybrid(name="hybrid_prompt", tokens=2000, snapshot=False),
        # the hybrid layers of one verify round in a graph, with a snapshot per token
        _hybrid(name="hybrid_verify", layers=12),
        # stochastic verify of 16 sequences through the output head
        _head(name="head_batch16", batch=16, temperature=0.7),
        # full-vocabulary acceptance of 16 sequences and the commit of their accepted rows
        dict(name="accept_general16", kind="general", drafts=3, batch=16, temperature=0.7, top_p=0.95),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("verify", "verify", "verify_batch", "tree", "prompt", "prompt", "round", "hybrid_verify",
                       "hybrid_prompt", "head", "general"))
    hq, hkv, d = rng.choice(GEOMETRIES)
    cache = rng.choice(("int8", "int8", "bf16"))
    geo = dict(q_heads=hq, kv_heads=hkv, head_dim=d, cache=cache)
    if kind == "verify":
        return _attn(**geo, tokens=rng.randint(1, 6), context=_log_int(rng, 64, 200000), outliers=rng.random() < 0.3,
                     out=rng.choice(("bf16", "bf16", "fp32")))
    if kind == "verify_batch":
        top = _log_int(rng, 512, 24576)
        return _attn(**geo, tokens=rng.randint(1, 5), batch=rng.randint(2, 16), context=top,
                     context_min=rng.randint(64, top // 2))
    if kind == "tree":
        top = _log_int(rng, 512, 65536)
        return _attn(**geo, tokens=rng.randint(5, 16), batch=rng.randint(1, 8), context=top,
                     context_min=rng.randint(64, top // 2), tree=True)
    if kind == "prompt":
        return _attn(**geo, tokens=_log_int(rng, 33, 2048 if d == 128 else 1280), context=rng.choice((0, _log_int(rng, 1, 2048))))
    if kind == "round":
        return dict(kind="round", layers=rng.randint(2, 16), context=_log_int(rng, 128, 16384), drafts=rng.randint(1, 5),
                    hidden=rng.choice((2048, 5120)))
    if kind == "hybrid_verify":
        return _hybrid(tokens=rng.randint(1, 6), layers=rng.randint(1, 12), value_heads=rng.choice((16, 32, 48)))
    if kind == "hybrid_prompt":
        return _hybrid(tokens=_log_int(rng, 33, 2000), snapshot=False, value_heads=rng.choice((16, 32, 48)))
    if kind == "head":
        return _head(hidden=rng.choice((2048, 5120)), batch=_log_int(rng, 1, 16), drafts=rng.randint(1, 3),
                     fused=rng.random() < 0.4, temperature=rng.choice((0.0, 0.7)))
    return dict(kind="general", drafts=rng.randint(1, 4), batch=_log_int(rng, 1, 12), temperature=rng.choice((0.6, 0.7, 1.0)),
                top_p=rng.choice((0.9, 0.95)))


# ---- inputs (plain torch, from the seed alone) -----------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _normal(g, shape, std=1.0, outliers=False):
    x = torch.randn(shape, generator=g, device=DEV, dtype=torch.float32)
    if outliers:  # one value in a hundred at +-20
        u = torch.rand(shape, generator=g, device=DEV)
        x = torch.where(u < 0.01, torch.where(u < 0.005, -20.0, 20.0), x)
    return (x * std).to(torch.bfloat16)


def _quantize(x):
    """INT8 group-64 codes and FP16 scales of BF16 rows [..., D]: s = FP16(amax / 127),
    code = clamp(rne(x * FP32(1 / s)), +-127)."""
    xf = x.float().unflatten(-1, (-1, 64))
    s = (xf.abs().amax(-1) / 127.0).half()
    inv = torch.where(s > 0, 1.0 / s.float(), 0.0)
    codes = (xf * inv[..., None]).round_().clamp_(-127, 127).to(torch.int8)
    return codes.flatten(-2), s


def _contexts(c):
    """History length of every sequence: part of the case, the same for every seed."""
    if c["batch"] == 1:
        return [c["context"]]
    r = random.Random(c["context"] * 31 + c["batch"])
    lo, hi = c["context_min"], c["context"]
    if c["tree"]:
        return [int(math.exp(r.uniform(math.log(lo), math.log(hi)))) for _ in range(c["batch"])]
    return [r.randint(lo, hi) for _ in range(c["batch"])]


def _padded(n):
    return (n + 127) // 128 * 128


def _cache_planes(g, c, B, P):
    """[B, Hkv, P, D] planes of a filled history (rows past it are overwritten or never visible)."""
    H, D = c["kv_heads"], c["head_dim"]
    k = torch.empty((B, H, P, D), device=DEV, dtype=torch.int8 if c["cache"] == "int8" else torch.bfloat16)
    v = torch.empty_like(k)
    if c["cache"] == "int8":
        ks = torch.empty((B, H, P, D // 64), device=DEV, dtype=torch.float16)
        vs = torch.empty_like(ks)
    for b in range(B):
        for h in range(H):
            for code, scale in ((k, 0), (v, 1)):
                x = _normal(g, (P, D), outliers=c.get("outliers", False))
                if c["cache"] == "int8":
                    q, s = _quantize(x)
                    code[b, h] = q
                    (vs if scale else ks)[b, h] = s
                else:
                    code[b, h] = x
    return (k, v, ks, vs) if c["cache"] == "int8" else (k, v)


def _attention_inputs(c, seed):
    g = _gen(seed)
    B, T, D = c["batch"], c["tokens"], c["head_dim"]
    Ls = _contexts(c)
    P = _padded(max(Ls) + T)
    d = dict(contexts=Ls, P=P, planes=_cache_planes(g, c, B, P))
    d["q"] = _normal(g, (B, T, c["q_heads"], D))
    d["k"] = _normal(g, (B, T, c["kv_heads"], D))
    d["v"] = _normal(g, (B, T, c["kv_heads"], D))
    d["base"] = torch.tensor(Ls, device=DEV, dtype=torch.int32)
    d["positions"] = (d["base"][:, None] + torch.arange(T, device=DEV, dtype=torch.int32)[None]).contiguous()
    if c["tree"]:
        d["parents"] = torch.tensor([[-1] + [(u - 1) // 2 for u in range(1, T)]] * B, device=DEV, dtype=torch.int32)
        r = random.Random(seed)
        target = [[r.randrange(VOCAB) for _ in range(T)] for _ in range(B)]
        node = [[0] + [t[(u - 1) // 2] if r.random() < 0.8 else r.randrange(VOCAB) for u in range(1, T)] for t in target]
        d["target"] = torch.tensor(target, device=DEV, dtype=torch.int32)
        d["node"] = torch.tensor(node, device=DEV, dtype=torch.int32)
    elif B > 1:
        d["keep"] = torch.randint(1, T + 1, (B,), generator=g, device=DEV, dtype=torch.int32)
    return d


def _q6_inputs(g, hidden):
    """A [VOCAB, hidden] Q6G64 RowSplit head: nibble, high-bit and scale planes in one payload."""
    G = (hidden + 127) // 128 * 2
    nb, hb, sb = VOCAB * G * 32, VOCAB * G * 16, VOCAB * G * 2
    hoff = (nb + 255) // 256 * 256
    soff = hoff + (hb + 255) // 256 * 256
    payload = torch.empty(soff + sb, device=DEV, dtype=torch.uint8)
    nib = payload[:nb].view(VOCAB, G, 32)
    high = payload[hoff:hoff + hb].view(VOCAB, G, 16)
    scale = payload[soff:].view(torch.float16).view(VOCAB, G)
    step = 31040
    for r in range(0, VOCAB, step):
        u = (torch.randn((step, G, 64), generator=g, device=DEV) * 10).round_().clamp_(-32, 31).to(torch.int16)
        u = (u & 63).to(torch.uint8)
        nib[r:r + step] = (u[..., 0::2] & 15) | ((u[..., 1::2] & 15) << 4)
        h = (u >> 4).view(step, G, 16, 4)
        high[r:r + step] = h[..., 0] | (h[..., 1] << 2) | (h[..., 2] << 4) | (h[..., 3] << 6)
        scale[r:r + step] = (torch.rand((step, G), generator=g, device=DEV) + 0.5).mul_(0.17 / math.sqrt(hidden)).half()
    return dict(payload=payload, nib=nib, high=high, scale=scale, hoff=hoff, soff=soff, hb=hb, G=G)


def _q6_logits64(w, x, hidden):
    """x [T, hidden] BF16 -> [T, VOCAB] in 64 bits."""
    out = torch.empty((x.shape[0], VOCAB), device=DEV, dtype=torch.float64)
    xt = torch.nn.functional.pad(x.double(), (0, w["G"] * 64 - hidden))
    step = 31040
    for r in range(0, VOCAB, step):
        nib, high = w["nib"][r:r + step], w["high"][r:r + step]
        low = torch.stack((nib & 15, nib >> 4), -1).flatten(-2)
        hi = torch.stack([(high >> (2 * m)) & 3 for m in range(4)], -1).flatten(-2)
        u = (low | (hi << 4)).to(torch.int16)
        code = torch.where(u >= 32, u - 64, u).double() * w["scale"][r:r + step].double()[..., None]
        out[:, r:r + step] = xt @ code.flatten(1).t().contiguous()
    return out


def _round_inputs(c, seed):
    g = _gen(seed)
    T = c["drafts"] + 1
    geo = _attn(context=c["context"], tokens=T)
    P = _padded(c["context"] + T)
    d = dict(P=P, planes=_cache_planes(g, geo, c["layers"], P), geo=geo)
    d["q"] = _normal(g, (c["layers"], T, 40, 128))
    d["k"] = _normal(g, (c["layers"], T, 8, 128))
    d["v"] = _normal(g, (c["layers"], T, 8, 128))
    d["x"] = _normal(g, (T, c["hidden"]))
    d["hidden"] = _normal(g, (T, c["hidden"]))
    d["w"] = _q6_inputs(g, c["hidden"])
    return d


def _hybrid_inputs(c, seed):
    g = _gen(seed)
    S, Hqk, Hv, T, n = c["head_dim"], c["qk_heads"], c["value_heads"], c["tokens"], c["layers"]
    C = 2 * Hqk * S + Hv * S
    silu = torch.nn.functional.silu
    rand = lambda *s: torch.rand(s, generator=g, device=DEV)  # noqa: E731
    d = dict(C=C, slots=T + 1 if c["snapshot"] else 0)
    # q, k, v as the layer's convolution leaves them; decay and step sizes of trained gated layers
    d["q"], d["k"] = (silu(_normal(g, (n, T, Hqk, S)).float()).to(torch.bfloat16) for _ in range(2))
    d["v"] = silu(_normal(g, (n, T, Hv, S)).float()).to(torch.bfloat16)
    d["g"] = -(1.0 + 15.0 * rand(n, 1, Hv)) * torch.exp(math.log(1e-3) + math.log(100.0) * rand(n, T, Hv))
    d["beta"] = torch.sigmoid(torch.randn((n, T, Hv), generator=g, device=DEV))
    d["x"] = _normal(g, (n, T, C))
    d["weight"] = _normal(g, (n, 4, C), 0.5)
    d["state"] = torch.randn((n, Hv, S, S), generator=g, device=DEV) * 0.05
    d["window"] = _normal(g, (n, 3, C))
    return d


# ---- views of torch memory -------------------------------------------------------------------

_DTYPES = {torch.bfloat16: na.BF16, torch.float32: na.FP32, torch.int32: na.I32, torch.int64: na.I64,
           torch.int8: na.I8, torch.float16: na.FP16}


def _view(t, shape=None):
    """nmi_tensor of a contiguous torch tensor (the package's order: fastest index first)."""
    return na.Tensor.make(t.data_ptr(), _DTYPES[t.dtype], shape or tuple(reversed(t.shape)))


def _kv_view(c, planes, max_context):
    """The layer view of planes [B, Hkv, P, D] (and scales)."""
    v = na.KVLayerView()
    v.k, v.v = _view(planes[0]), _view(planes[1])
    if len(planes) == 4:
        v.k_scale, v.v_scale = _view(planes[2]), _view(planes[3])
    v.max_context, v.padded_context = max_context, planes[0].shape[2]
    v.num_kv_heads, v.head_dim = c["kv_heads"], c["head_dim"]
    v.dtype = na.I8 if len(planes) == 4 else na.BF16
    v.quant_group = 64 if len(planes) == 4 else 0
    return v


def _q6_view(w, hidden):
    r = na.Weight()
    p = w["payload"].data_ptr()
    r.payload, r.payload_bytes, r.high_plane_bytes = p, w["payload"].numel(), w["hb"]
    r.qtype, r.group_size, r.ndim = 2, 64, 2
    r.shape[:] = [VOCAB, hidden, 1, 1]
    r.padded_shape[:] = [VOCAB, w["G"] * 64, 1, 1]
    r.qdata, r.qhigh, r.scales = p, p + w["hoff"], p + w["soff"]
    r.n, r.k, r.group, r.layout, r.scale_dtype = VOCAB, hidden, 64, 0, na.FP16
    return r


def _i32(*shape):
    return torch.zeros(shape, device=DEV, dtype=torch.int32)


def _sampling_configs(temperature, batch, seed):
    blob = b""
    for b in range(batch):
        cfg = na.SamplingConfig()
        if temperature > 0:
            cfg.temperature, cfg.top_p, cfg.seed = temperature, 0.95, (int(seed) * 1000 + b) & 0x7FFFFFFFFFFFFFFF
        blob += bytes(memoryview(cfg))
    return torch.frombuffer(bytearray(blob), dtype=torch.uint8).to(DEV)


def _accept_state(B, K, length):
    """Device scalars of an acceptance round and their views."""
    t = dict(drafts=_i32(B, K), length=_i32(B) + length, token=_i32(B), sampled=_i32(B, K + 1), num=_i32(B),
             accepted=_i32(B), stats=torch.zeros((B, 4 + K), device=DEV, dtype=torch.int64))
    return t


def _plant_drafts(x, w, hidden, B, K, seed):
    """Drafts as a good draft model leaves them: the target's argmax, one in five replaced."""
    T = B * (K + 1)
    target = _i32(T)
    ws = DeviceBuffer(ops.linear_argmax_workspace_bytes(T))
    ops.linear_argmax(_view(x, (hidden, T)), _q6_view(w, hidden), VOCAB, ws, _view(target))
    torch.cuda.synchronize()
    r = random.Random(seed)
    rows = target.view(B, K + 1)[:, :K].tolist()
    rows = [[t if r.random() < 0.8 else r.randrange(VOCAB) for t in row] for row in rows]
    return torch.tensor(rows, device=DEV, dtype=torch.int32).view(B, K)


# ---- prepare ---------------------------------------------------------------------------------

def prepare(case, seed):
    s = {"attention": _prepare_attention, "round": _prepare_round, "hybrid": _prepare_hybrid, "head": _prepare_head,
         "general": _prepare_general}[case["kind"]](case, seed)
    torch.cuda.synchronize()
    return s


def _prepare_attention(c, seed):
    d = _attention_inputs(c, seed)
    B, T, D = c["batch"], c["tokens"], c["head_dim"]
    max_context = max(d["contexts"]) + T
    out = torch.zeros((B, T, c["q_heads"], D), device=DEV, dtype=torch.float32 if c["out"] == "fp32" else torch.bfloat16)
    need = ops.gqa_attention_workspace_bytes(c["q_heads"], c["kv_heads"], D, T, B, max_context)
    s = dict(case=c, keep_alive=d, out=out, ws=DeviceBuffer(max(256, need)), cache=_kv_view(c, d["planes"], max_context),
             scale=1.0 / math.sqrt(D), envelope=(min(d["contexts"]) + (T if T <= 32 else 1), max_context))
    s["views"] = {n: _view(d[n]) for n in ("q", "k", "v", "positions")}
    s["views"]["out"] = _view(out)
    s["outputs"] = [out, *d["planes"]]
    if c["tree"]:
        t = dict(path=_i32(B, T), path_len=_i32(B), length=d["base"].clone(), token=_i32(B), sampled=_i32(B, T), num=_i32(B),
                 accepted=_i32(B), stats=torch.zeros((B, 4 + T), device=DEV, dtype=torch.int64))
        s["views"].update({n: _view(d[n]) for n in ("parents", "node", "target", "base")})
        s["views"].update({n: _view(x) for n, x in t.items()})
        s["outputs"] += [t[n] for n in ("path", "path_len", "length", "token", "sampled", "num", "accepted", "stats")]
        s["tree"] = t
    elif B > 1 and c["cache"] == "int8":
        s["views"]["keep"] = _view(d["keep"])
    return s


def _prepare_round(c, seed):
    d = _round_inputs(c, seed)
    K, T, n = c["drafts"], c["drafts"] + 1, c["layers"]
    L = c["context"]
    t = _accept_state(1, K, L)
    t["drafts"] = _plant_drafts(d["x"], d["w"], c["hidden"], 1, K, seed)
    t.update(start=_i32(1) + L, ids=_i32(T), positions=_i32(T), target=_i32(T), align=_i32(T), slot=_i32(1),
             selected=torch.zeros((1, c["hidden"]), device=DEV, dtype=torch.bfloat16),
             logits=torch.zeros((T, VOCAB), device=DEV, dtype=torch.bfloat16), out=torch.zeros_like(d["q"]))
    t["token"] += 7
    ws = DeviceBuffer(max(256, ops.gqa_attention_workspace_bytes(40, 8, 128, T, 1, L + T)))
    ws_accept = DeviceBuffer(max(256, ops.sampling_workspace_bytes(VOCAB, T, 1)))
    cfg = _sampling_configs(0.0, 1, seed)
    weight = _q6_view(d["w"], c["hidden"])
    caches = [_kv_view(d["geo"], [p[i:i + 1] for p in d["planes"]], L + T) for i in range(n)]
    layer = [[_view(x[i:i + 1]) for x in (d["q"], d["k"], d["v"], t["out"])] for i in range(n)]
    v = {k: _view(x) for k, x in t.items()}
    # one sequence: scalars [1], ids and positions [T], drafts [K], logits [rows, T], stats [4 + K]
    v.update(drafts=_view(t["drafts"], (K,)), sampled=_view(t["sampled"], (T,)), stats=_view(t["stats"], (4 + K,)))
    x, hidden = _view(d["x"]), _view(d["hidden"])
    torch.cuda.synchronize()
    stream = Stream()
    with Graph(stream) as graph:
        ops.assign_i32_scalar(v["start"], v["length"], stream)
        ops.speculative_prepare_verify_inputs(v["token"], v["drafts"], v["length"], v["ids"], v["positions"], stream)
        for (q, k, vv, out), cache in zip(layer, caches):
            ops.gqa_attention(q, k, vv, v["positions"], 1.0 / math.sqrt(128), cache, (L + T, L + T), ws, out, stream)
        ops.linear(x, weight, v["logits"], stream)
        ops.argmax(v["logits"], v["target"], VOCAB, stream)
        ops.speculative_accept_greedy_drafts(v["target"], v["logits"], v["drafts"], v["length"], v["token"], v["sampled"],
                                             v["num"], v["accepted"], v["stats"], VOCAB, cfg.data_ptr(), ws_accept, stream)
        ops.speculative_select_accepted_hidden(hidden, v["accepted"], v["selected"], stream)
        ops.mtp_prepare_alignment_ids(v["ids"], v["token"], v["accepted"], v["align"], stream)
        ops.assign_i32_scalar(v["accepted"], v["slot"], stream)
    outputs = [t["out"], t["logits"], t["selected"], *d["planes"]]
    outputs += [t[k] for k in ("target", "length", "token", "sampled", "num", "accepted", "stats", "slot")]
    # alignment ids past the accepted slot are not written: they are not part of the result
    return dict(case=c, graph=graph, stream=stream, outputs=outputs, keep_alive=(d, t, ws, ws_accept, cfg))


def _prepare_hybrid(c, seed):
    d = _hybrid_inputs(c, seed)
    S, Hqk, Hv, T, n, C = c["head_dim"], c["qk_heads"], c["value_heads"], c["tokens"], c["layers"], d["C"]
    t = dict(conv=torch.zeros_like(d["x"]), out=torch.zeros_like(d["v"]))
    scale = 1.0 / math.sqrt(S)
    s = dict(case=c, keep_alive=(d, t))
    calls = []
    if c["snapshot"]:
        # the accepted state of the last round sits in the slot past those this round writes
        t["states"] = torch.zeros((n, T + 1, Hv, S, S), device=DEV)
        t["windows"] = torch.zeros((n, T + 1, 3, C), device=DEV, dtype=torch.bfloat16)
        t["states"][:, T] = d["state"]
        t["windows"][:, T] = d["window"]
        slot = _i32(1) + T
        t["slot"] = slot
        for i in range(n):
            calls.append((ops.causal_conv1d_silu_snapshot,
                          (_view(d["x"][i]), _view(d["weight"][i]), _view(t["windows"][i]), _view(slot), _view(t["conv"][i]))))
            calls.append((ops.gated_delta_rule_snapshot,
                          (_view(d["q"][i]), _view(d["k"][i]), _view(d["v"][i]), _view(d["g"][i]), _view(d["beta"][i]), scale,
                           True, _view(t["states"][i]), _view(slot), _view(t["out"][i]))))
        s["outputs"] = [t["conv"], t["out"], t["states"], t["windows"]]
    else:
        t["state_out"] = torch.zeros_like(d["state"])
        t["window_out"] = torch.zeros_like(d["window"])
        for i in range(n):
            calls.append((ops.causal_conv1d_silu,
                          (_view(d["x"][i]), _view(d["weight"][i]), _view(d["window"][i]), _view(t["window_out"][i]),
                           _view(t["conv"][i]))))
            calls.append((ops.gated_delta_rule,
                          (_view(d["q"][i]), _view(d["k"][i]), _view(d["v"][i]), _view(d["g"][i]), _view(d["beta"][i]), scale,
                           True, _view(d["state"][i]), _view(t["state_out"][i]), _view(t["out"][i]))))
        s["outputs"] = [t["conv"], t["out"], t["state_out"], t["window_out"]]
    if n > 1:  # a round's layers are captured once
        torch.cuda.synchronize()
        s["stream"] = Stream()
        with Graph(s["stream"]) as graph:
            for fn, args in calls:
                fn(*args, s["stream"])
        s["graph"] = graph
    else:
        s["calls"] = calls
    return s


def _prepare_head(c, seed):
    g = _gen(seed)
    K, B, H = c["drafts"], c["batch"], c["hidden"]
    T = B * (K + 1)
    w = _q6_inputs(g, H)
    x = _normal(g, (B, K + 1, H))
    t = _accept_state(B, K, 600)
    t["drafts"] = _plant_drafts(x, w, H, B, K, seed)
    t["target"] = _i32(B, K + 1)
    cfg = _sampling_configs(c["temperature"], B, seed)
    s = dict(case=c, weight=_q6_view(w, H), cfg=cfg.data_ptr(), views={k: _view(v) for k, v in t.items()})
    s["outputs"] = [t[k] for k in ("length", "token", "sampled", "num", "accepted", "stats")]
    if c["fused"]:
        s["views"]["x"] = _view(x)
        s["ws"] = DeviceBuffer(ops.speculative_accept_fused_head_workspace_bytes(K, B))
    else:
        t["logits"] = torch.zeros((B, K + 1, VOCAB), device=DEV, dtype=torch.bfloat16)
        s["views"].update(x=_view(x, (H, T)), logits=_view(t["logits"]), columns=_view(t["logits"], (VOCAB, T)))
        s["ws"] = DeviceBuffer(max(256, ops.sampling_workspace_bytes(VOCAB, K + 1, B)))
        s["outputs"] = [t["logits"], *s["outputs"]]
    s["keep_alive"] = (w, x, t, cfg)
    return s


def _prepare_general(c, seed):
    g = _gen(seed)
    K, B = c["drafts"], c["batch"]
    t = _accept_state(B, K, 4096)
    std = math.sqrt(3.0)
    target = torch.randn((B, K + 1, VOCAB), generator=g, device=DEV) * std
    draft = 0.9 * target[:, :K] + math.sqrt(1 - 0.81) * std * torch.randn((B, K, VOCAB), generator=g, device=DEV)
    t["logits"], t["draft_logits"] = target.to(torch.bfloat16), draft.to(torch.bfloat16)
    # drafts sampled from the draft model at the same temperature (Gumbel maximum)
    noise = -torch.log(-torch.log(torch.rand(draft.shape, generator=g, device=DEV).clamp_(1e-12, 1 - 1e-7)))
    t["drafts"] = (t["draft_logits"].float() / c["temperature"] + noise).argmax(-1).to(torch.int32)
    del target, draft, noise
    t["u_accept"] = torch.rand((B, K + 1), generator=g, device=DEV)
    t["u_residual"] = torch.rand((B, 1), generator=g, device=DEV)
    cfg = torch.tensor([c["temperature"], c["top_p"]], device=DEV, dtype=torch.float32)
    # the accepted rows' K/V go to rows 256.. of every sequence's cache
    geo = _attn(batch=B, context=256, tokens=K + 1)
    planes = _cache_planes(g, geo, B, 384)
    k, v = _normal(g, (B, K + 1, 8, 128)), _normal(g, (B, K + 1, 8, 128))
    pos = (256 + torch.arange(K + 1, device=DEV, dtype=torch.int32)).repeat(B, 1).contiguous()
    views = {n: _view(x) for n, x in t.items()}
    views.update(k=_view(k), v=_view(v), positions=_view(pos))
    return dict(case=c, views=views, cfg=cfg.data_ptr(), cache=_kv_view(geo, planes, 384),
                ws=DeviceBuffer(max(256, ops.general_accept_workspace_bytes(VOCAB, K, B))),
                outputs=[*(t[n] for n in ("length", "token", "sampled", "num", "accepted", "stats")), *planes],
                keep_alive=(t, cfg, planes, k, v, pos))


# ---- run -------------------------------------------------------------------------------------

def run(state):
    kind = state["case"]["kind"]
    if "graph" in state:
        state["graph"].launch()
    elif kind == "attention":
        _run_attention(state)
    elif kind == "hybrid":
        for fn, args in state["calls"]:
            fn(*args)
    elif kind == "head":
        _run_head(state)
    else:
        v, K = state["views"], state["case"]["drafts"]
        ops.speculative_accept_general(v["logits"], v["draft_logits"], v["drafts"], v["u_accept"], v["u_residual"], v["length"],
                                       v["token"], v["sampled"], v["num"], v["accepted"], v["stats"], VOCAB, state["cfg"],
                                       state["ws"])
        ops.kv_cache_append_prefix(v["k"], v["v"], v["positions"], v["num"], (1, K + 1), state["cache"])
    return state["outputs"]


def _run_attention(s):
    c, v = s["case"], s["views"]
    if c["tree"]:
        ops.gqa_attention_tree(v["q"], v["k"], v["v"], v["positions"], v["parents"], s["scale"], s["cache"], s["envelope"],
                               True, s["ws"], v["out"])
        ops.tree_accept_greedy(v["parents"], v["node"], v["target"], v["path"], v["path_len"], v["length"], v["token"],
                               v["sampled"], v["num"], v["accepted"], v["stats"])
        if c["cache"] == "int8":
            ops.kv_cache_compact_path(v["base"], v["path"], v["path_len"], s["cache"])
        return
    ops.gqa_attention(v["q"], v["k"], v["v"], v["positions"], s["scale"], s["cache"], s["envelope"], s["ws"], v["out"])
    if "keep" in v:
        ops.kv_cache_rollback(v["positions"], v["keep"], s["cache"])


def _run_head(s):
    c, v = s["case"], s["views"]
    if c["fused"]:
        ops.speculative_accept_fused_head(v["x"], s["weight"], v["drafts"], v["length"], v["token"], v["sampled"], v["num"],
                                          v["accepted"], v["stats"], VOCAB, s["cfg"], s["ws"])
        return
    ops.linear(v["x"], s["weight"], v["columns"])
    if c["temperature"] <= 0:
        ops.argmax(v["logits"], v["target"], VOCAB)
    ops.speculative_accept_greedy_drafts(v["target"], v["logits"], v["drafts"], v["length"], v["token"], v["sampled"],
                                         v["num"], v["accepted"], v["stats"], VOCAB, s["cfg"], s["ws"])


# ---- what a pass cannot do without -----------------------------------------------------------

def _attention_work(c, Ls):
    D, T, Hq, Hkv = c["head_dim"], c["tokens"], c["q_heads"], c["kv_heads"]
    row = 2 * Hkv * (D + 2 * (D // 64)) if c["cache"] == "int8" else 4 * Hkv * D  # K and V of one key
    nbytes = flops = 0
    for L in Ls:
        nbytes += (L + T) * row  # history read, new rows written
        nbytes += T * Hq * D * (2 + (4 if c["out"] == "fp32" else 2)) + 2 * T * Hkv * D * 2
        flops += 4 * D * Hq * (T * L + T * (T + 1) // 2)
    return nbytes, flops


def work(case):
    c, kind = case, case["kind"]
    if kind == "attention":
        b, f = _attention_work(c, _contexts(c))
        return {"bytes": b, "flops": f}
    if kind == "round":
        T = c["drafts"] + 1
        b, f = _attention_work(_attn(tokens=T, context=c["context"]), [c["context"]])
        G = (c["hidden"] + 127) // 128 * 2
        return {"bytes": c["layers"] * b + VOCAB * G * 50 + T * (c["hidden"] * 2 + VOCAB * 2),
                "flops": c["layers"] * f + 2 * T * VOCAB * c["hidden"]}
    if kind == "hybrid":
        S, Hqk, Hv, T = c["head_dim"], c["qk_heads"], c["value_heads"], c["tokens"]
        C = 2 * Hqk * S + Hv * S
        slots = T if c["snapshot"] else 1
        b = S * S * Hv * 4 * (1 + slots) + T * (2 * S * Hqk * 2 + 2 * S * Hv * 2 + 2 * Hv * 4) + C * 2 * (3 + 3 * slots + 2 * T + 4)
        return {"bytes": c["layers"] * b, "flops": c["layers"] * T * (Hv * S * S * 7 + C * 12)}
    if kind == "head":
        T = c["batch"] * (c["drafts"] + 1)
        G = (c["hidden"] + 127) // 128 * 2
        return {"bytes": VOCAB * G * 50 + T * c["hidden"] * 2 + (0 if c["fused"] else T * VOCAB * 2),
                "flops": 2 * T * VOCAB * c["hidden"]}
    cols = (2 * c["drafts"] + 1) * c["batch"]
    return {"bytes": cols * VOCAB * 2, "flops": 0}


def tolerance(case):
    """Relative 2-norm differences between correct implementations at the same precision. Attention
    operands are 16-bit (rounded once) and the usual output BF16: the present code is 1.7e-3 from 64
    bits with BF16 results and 4e-4 with FP32 ones. The head's logits are FP32 sums rounded to BF16
    (1.7e-3), the recurrence FP32 with BF16 outputs (1.7e-3)."""
    kind = case["kind"]
    if kind == "general":
        return "exact"
    if kind == "attention" and case["out"] == "fp32":
        return {"rel": 2e-3}
    return {"rel": 7e-3}


# ---- the same results in 64 bits, in plain torch ----------------------------------------------

def _attention64(q, k, v, planes, L, parents):
    """One sequence: q [T, Hq, D], new k/v [T, Hkv, D], planes of that sequence [Hkv, P, ...]."""
    T, Hq, D = q.shape
    H = k.shape[1]
    G = Hq // H
    out = torch.empty((T, Hq, D), device=DEV, dtype=torch.float64)
    see = torch.ones((T, T), device=DEV, dtype=torch.bool).tril()
    if parents is not None:
        see = torch.eye(T, device=DEV, dtype=torch.bool)
        for u in range(1, T):
            see[u] |= see[int(parents[u])]
    if len(planes) == 4:
        dequantize = lambda codes, s: (codes.double().unflatten(-1, (-1, 64)) * s.double()[..., None]).flatten(-2)  # noqa: E731
        (kc, ks), (vc, vs) = _quantize(k), _quantize(v)
        nk, nv = dequantize(kc, ks), dequantize(vc, vs)
    else:
        nk, nv = k.double(), v.double()
    for h in range(H):
        if len(planes) == 4:
            hk, hv = dequantize(planes[0][h, :L], planes[2][h, :L]), dequantize(planes[1][h, :L], planes[3][h, :L])
        else:
            hk, hv = planes[0][h, :L].double(), planes[1][h, :L].double()
        kk, vv = torch.cat((hk, nk[:, h])), torch.cat((hv, nv[:, h]))
        qq = q[:, h * G:(h + 1) * G].double().reshape(T * G, D)
        score = (qq @ kk.t().contiguous()).div_(math.sqrt(D))
        score[:, L:].masked_fill_(~see.repeat_interleave(G, 0), -math.inf)
        out[:, h * G:(h + 1) * G] = (torch.softmax(score, -1) @ vv).view(T, G, D)
    return out


def _hybrid64(c, d, i):
    """Layer i: conv out [T, C], recurrence out [T, Hv, S], states [T, Hv, S, S], windows [T, 3, C]."""
    S, Hqk, Hv, T = c["head_dim"], c["qk_heads"], c["value_heads"], c["tokens"]
    u = torch.cat((d["window"][i], d["x"][i])).double()
    y = sum(d["weight"][i, j].double() * u[j:j + T] for j in range(4))
    conv = y * torch.sigmoid(y)
    q, k = d["q"][i].double(), d["k"][i].double()
    q = (q / (q.square().sum(-1, keepdim=True) + 1e-6).sqrt()).repeat_interleave(Hv // Hqk, 1)
    k = (k / (k.square().sum(-1, keepdim=True) + 1e-6).sqrt()).repeat_interleave(Hv // Hqk, 1)
    v, alpha, beta = d["v"][i].double(), d["g"][i].double().exp(), d["beta"][i].double()
    st = d["state"][i].double()
    outs, states = [], []
    for t in range(T):
        st = st * alpha[t, :, None, None]
        delta = beta[t, :, None] * (v[t] - (st * k[t, :, None, :]).sum(-1))
        st = st + delta[..., None] * k[t, :, None, :]
        outs.append((st * q[t, :, None, :]).sum(-1) / math.sqrt(S))
        if c["snapshot"] or t == T - 1:
            states.append(st)
    windows = torch.stack([u[t + 1:t + 4] for t in (range(T) if c["snapshot"] else (T - 1,))])
    return conv, torch.stack(outs), torch.stack(states), windows


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "attention":
        if c["tokens"] * (max(_contexts(c)) + c["tokens"]) * c["q_heads"] * c["batch"] > 1 << 31:
            return None
        d = _attention_inputs(c, seed)
        out = torch.stack([_attention64(d["q"][b], d["k"][b], d["v"][b], [p[b] for p in d["planes"]], L,
                                        d["parents"][b] if c["tree"] else None) for b, L in enumerate(d["contexts"])])
        return [out] + [None] * (len(d["planes"]) + (8 if c["tree"] else 0))
    if kind == "round":
        d = _round_inputs(c, seed)
        out = torch.stack([_attention64(d["q"][i], d["k"][i], d["v"][i], [p[i] for p in d["planes"]], c["context"], None)
                           for i in range(c["layers"])])
        return [out, _q6_logits64(d["w"], d["x"], c["hidden"])] + [None] * 13
    if kind == "hybrid":
        d = _hybrid_inputs(c, seed)
        conv, outs, states, windows = (list(x) for x in zip(*(_hybrid64(c, d, i) for i in range(c["layers"]))))
        if not c["snapshot"]:
            return [torch.stack(conv), torch.stack(outs), torch.cat(states), torch.cat(windows)]
        last = [torch.cat((s, d["state"][i][None].double())) for i, s in enumerate(states)]
        lastw = [torch.cat((w, d["window"][i][None].double())) for i, w in enumerate(windows)]
        return [torch.stack(conv), torch.stack(outs), torch.stack(last), torch.stack(lastw)]
    if kind == "head" and not c["fused"]:
        g = _gen(seed)
        w = _q6_inputs(g, c["hidden"])
        x = _normal(g, (c["batch"], c["drafts"] + 1, c["hidden"]))
        return [_q6_logits64(w, x.flatten(0, 1), c["hidden"]).view(c["batch"], c["drafts"] + 1, VOCAB)] + [None] * 6
    return None
