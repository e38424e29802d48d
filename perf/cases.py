"""The work that programs have this package do, as cases that can be timed and checked.

Shapes are those of the configurations in ``qvex.model.Config`` (the 9B text
shape and the tiny one): 4-bit group-64 weights, 24 Gated DeltaNet layers and 8
gated attention layers, prompts in 512-token chunks, verify calls of k + 1 rows.
A decode-side call (1..8 rows) is captured once as a HIP graph and replayed, as
``speculative.decode()`` runs it; the prompt-side calls are launched eagerly, as
``engine.prefill`` runs them.

Kinds: ``linear`` (QLinear), ``mlp`` (MLP), ``gdn`` and ``attn`` (the two
mixers), ``layer`` (a decoder layer of a verify call), ``accept`` (the acceptance
sampler), ``draft`` (one MTP head step), ``verify`` and ``prefill`` (the whole
model).
"""

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "qvex-3.5_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from qvex import kernels  # noqa: E402
from qvex.engine import prefill  # noqa: E402
from qvex.model import (MLP, Attention, CacheCounters, Config, GatedDeltaNet, KVCache, Layer, NormedRows, QEmbedding,  # noqa: E402
                        QLinear, Qwen35, RecurrentCache, random_model)
from qvex.mtp import MTPHead, random_mtp  # noqa: E402

DEV = "cuda:0"
BF16 = torch.bfloat16
VOCAB = 248320
WIDTH = 8            # widest verify call (make_cache's default)
CHUNK = 512          # prompt tokens per forward call
MAX_CONTEXT = 8192   # the default KV capacity


def listed():
    return [
        # one draft step of the decode cycle: the MTP head and the vocabulary-wide lm_head on one row
        {"name": "draft_1", "kind": "draft", "shape": "9b", "ctx": 4096},
        # the verify call of the k = 3 decode cycle: all 32 layers and the lm_head on 4 rows
        {"name": "verify_4", "kind": "verify", "shape": "9b", "rows": 4, "ctx": 4096},
        # one DeltaNet layer and one attention layer of a verify call
        {"name": "layer_gdn_verify_4", "kind": "layer", "shape": "9b", "linear": True, "rows": 4, "ctx": 4096},
        {"name": "layer_attn_verify_6", "kind": "layer", "shape": "9b", "linear": False, "rows": 6, "ctx": 7001},
        # the ragged last chunk of a prompt through the attention input projection
        {"name": "linear_tail_37", "kind": "linear", "rows": 37, "n": 10240, "k": 4096, "bits": 4, "group": 64},
        # a prompt's tail through a module that the quantization config keeps at 8 bits
        {"name": "linear_8bit_200", "kind": "linear", "rows": 200, "n": 4096, "k": 4096, "bits": 8, "group": 64},
        # one 512-token prompt chunk through the MLP and through each mixer
        {"name": "mlp_prefill_512", "kind": "mlp", "shape": "9b", "rows": 512},
        {"name": "gdn_prefill_512", "kind": "gdn", "shape": "9b", "rows": 512, "ctx": 1024},
        {"name": "attn_prefill_512", "kind": "attn", "shape": "9b", "rows": 512, "ctx": 3584},
        # acceptance of one verify call as decode() samples it, and of 256 steps with draft logits
        {"name": "accept_1_k3", "kind": "accept", "steps": 1, "drafts": 3, "vocab": VOCAB, "draft_logits": False,
         "temperature": 0.7, "top_k": 20, "top_p": 0.8},
        {"name": "accept_256_k4", "kind": "accept", "steps": 256, "drafts": 4, "vocab": VOCAB, "draft_logits": True,
         "temperature": 0.7, "top_k": 0, "top_p": 1.0},
        # a whole prompt: 2048 tokens in 512-token chunks, the MTP head fed as it goes
        {"name": "prefill_2048", "kind": "prefill", "shape": "9b", "rows": 2048},
    ]


def _loguniform(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "mlp", "gdn", "gdn", "attn", "attn", "layer", "layer", "accept",
                       "accept", "draft"])
    shape = rng.choice(["9b", "9b", "9b", "tiny"])
    if kind == "linear":
        bits = rng.choice([4, 4, 4, 4, 3, 5, 6, 8])
        group = 64 if bits == 4 else rng.choice([32, 64, 128])
        k = rng.choice([512, 1024, 2048, 4096, 4096, 8192, 12288, 128 * rng.randint(2, 64)])
        n = rng.choice([4096, 10240, 12352, 24576, _loguniform(rng, 64, 24576), 8 * _loguniform(rng, 8, 3072)])
        return {"kind": "linear", "rows": _loguniform(rng, 1, 1024), "n": n, "k": k, "bits": bits, "group": group}
    if kind == "mlp":
        return {"kind": "mlp", "shape": shape, "rows": _loguniform(rng, 1, 1024)}
    if kind in ("gdn", "attn"):
        rows = _loguniform(rng, 1, CHUNK)
        rows += kind == "gdn" and rows % (WIDTH + 1) == 0   # a pass leaves the state it starts from in place
        ctx = rng.choice([0, _loguniform(rng, 16, 16384)])
        return {"kind": kind, "shape": shape, "rows": min(rows, CHUNK), "ctx": ctx}
    if kind == "layer":
        return {"kind": "layer", "shape": shape, "linear": rng.random() < 0.5, "rows": rng.randint(1, WIDTH),
                "ctx": _loguniform(rng, 16, 16384)}
    if kind == "draft":
        return {"kind": "draft", "shape": shape, "ctx": _loguniform(rng, 16, 16384)}
    v = rng.choice([VOCAB, VOCAB, 4 * _loguniform(rng, 512, 62080)])
    filtered = rng.random() < 0.5
    return {"kind": "accept", "steps": _loguniform(rng, 1, 128), "drafts": rng.randint(1, 7), "vocab": v,
            "draft_logits": not filtered and rng.random() < 0.5, "temperature": rng.choice([0.0, 0.6, 0.7, 1.0]),
            "top_k": 20 if filtered else 0, "top_p": rng.choice([0.8, 0.95]) if filtered else 1.0}


# ---------------------------------------------------------------- inputs

def _cfg(shape, layers=None):
    cfg = Config.qwen35_9b() if shape == "9b" else Config.tiny()
    if layers is not None:
        cfg.num_hidden_layers = layers
    return cfg


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(1_000_003 * int(seed) + 17)
    return g


def _rows(g, m, k, scale=1.0):
    return (torch.randn((m, k), generator=g, device=DEV) * scale).to(BF16)


def _norm_w(g, n):
    return (1.0 + 0.1 * torch.randn(n, generator=g, device=DEV)).to(BF16)


def _affine(g, n, k, bits=4, group=64, gain=1.0):
    """Codes uniform, dequantized weights of zero mean and variance gain^2 / K: (w, scales, biases, bits, group)."""
    w = torch.randint(-2 ** 31, 2 ** 31, (n, k * bits // 32), generator=g, device=DEV, dtype=torch.int64).to(torch.int32)
    step = gain / math.sqrt((4 ** bits - 1) / 12 * k)
    s = ((torch.rand((n, k // group), generator=g, device=DEV) + 0.5) * step).to(BF16)
    b = (-(2 ** (bits - 1)) * s.float()).to(BF16)
    return w, s, b, bits, group


def _qlinear(a):
    w, s, b, bits, group = a
    return QLinear(w, s, b, group, bits)


def _mlp_raw(g, cfg):
    H, I = cfg.hidden_size, cfg.intermediate_size
    return {"gate_proj": _affine(g, I, H), "up_proj": _affine(g, I, H), "down_proj": _affine(g, H, I, gain=0.5)}


def _gdn_raw(g, cfg):
    H = cfg.hidden_size
    kd = cfg.linear_num_key_heads * cfg.linear_key_head_dim
    vd = cfg.linear_num_value_heads * cfg.linear_value_head_dim
    hv = cfg.linear_num_value_heads
    return {"in_proj_qkv": _affine(g, 2 * kd + vd, H), "in_proj_z": _affine(g, vd, H), "in_proj_b": _affine(g, hv, H),
            "in_proj_a": _affine(g, hv, H), "out_proj": _affine(g, H, vd, gain=0.5),
            "conv1d": (0.5 * torch.randn((2 * kd + vd, cfg.linear_conv_kernel_dim), generator=g, device=DEV)).to(BF16),
            "A_log": 0.5 * torch.randn(hv, generator=g, device=DEV),
            "dt_bias": (0.5 * torch.randn(hv, generator=g, device=DEV)).to(BF16),
            "norm": _norm_w(g, cfg.linear_value_head_dim)}


def _attn_raw(g, cfg):
    H, D = cfg.hidden_size, cfg.head_dim
    hq, hkv = cfg.num_attention_heads, cfg.num_key_value_heads
    return {"q_proj": _affine(g, 2 * hq * D, H), "k_proj": _affine(g, hkv * D, H), "v_proj": _affine(g, hkv * D, H),
            "o_proj": _affine(g, H, hq * D, gain=0.5), "q_norm": _norm_w(g, D), "k_norm": _norm_w(g, D)}


def _layers_of(raw):
    return {k: _qlinear(v) if isinstance(v, tuple) else v for k, v in raw.items()}


def _gdn_state(g, cfg, ctx):
    """The three conv rows before position ctx and the DeltaNet state there (zero at the start of a prompt)."""
    kd = cfg.linear_num_key_heads * cfg.linear_key_head_dim
    vd = cfg.linear_num_value_heads * cfg.linear_value_head_dim
    on = 1.0 if ctx else 0.0
    conv = _rows(g, cfg.linear_conv_kernel_dim - 1, 2 * kd + vd, on)
    state = 0.02 * on * torch.randn((cfg.linear_num_value_heads, cfg.linear_value_head_dim, cfg.linear_key_head_dim),
                                    generator=g, device=DEV)
    return conv, state


def _gdn_cache(cfg, mixer, ctx, conv, state):
    counters = CacheCounters(1, DEV)
    c = RecurrentCache(counters, 0, conv_dim=mixer.conv_dim, kernel=mixer.K, hv=mixer.hv, dv=mixer.dv, dk=mixer.dk,
                       max_width=WIDTH, device=DEV, prefill_width=CHUNK)
    rows = [(ctx - conv.shape[0] + j) % c.ring_rows for j in range(conv.shape[0])]
    c.conv_ring[rows] = conv
    c.ssm_ring[ctx % c.n_slots, 0] = state
    c.offset = ctx
    counters.sync()
    return c


def _kv_state(g, cfg, ctx):
    """Normalised keys and values of ctx earlier positions, [Hkv, ctx, D]."""
    shape = (cfg.num_key_value_heads, ctx, cfg.head_dim)
    return (torch.randn(shape, generator=g, device=DEV).to(BF16), torch.randn(shape, generator=g, device=DEV).to(BF16))


def _tile_k(k):
    h, cap, D = k.shape
    return k.reshape(h, cap // 16, 16, D // 32, 4, 8).permute(0, 1, 3, 4, 2, 5).reshape(h, cap // 16, D // 32, 64, 8)


def _tile_v(v):
    h, cap, D = v.shape
    return v.reshape(h, cap // 32, 32, D).permute(0, 1, 3, 2)


def _capacity(ctx, rows):
    return max(MAX_CONTEXT, (ctx + rows + 255) // 256 * 256)


def _padded(x, cap):
    out = torch.zeros((x.shape[0], cap, x.shape[2]), dtype=x.dtype, device=x.device)
    out[:, :x.shape[1]] = x
    return out


def _kv_cache(cfg, ctx, rows, k, v):
    c = KVCache(None, 0, n_kv=cfg.num_key_value_heads, head_dim=cfg.head_dim, capacity=_capacity(ctx, rows), device=DEV)
    if ctx:
        c.k.copy_(_tile_k(_padded(k, c.capacity)).view_as(c.k))
        c.v.copy_(_tile_v(_padded(v, c.capacity)))
    c.offset = ctx
    c.counters.sync()
    return c


def _captured(counters, body):
    """`body` run once, then recorded as a HIP graph that leaves the position counters where they are."""
    host = counters.host.copy()

    def back():
        counters.host[:] = host

    body()
    back()
    torch.cuda.synchronize()
    counters.graph_mode = counters.capturing = True
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = body()
    counters.capturing = False
    back()
    return graph, out


def _linear_inputs(case, seed):
    g = _gen(seed)
    return _affine(g, case["n"], case["k"], case["bits"], case["group"]), _rows(g, case["rows"], case["k"])


def _mlp_inputs(case, seed):
    g, cfg = _gen(seed), _cfg(case["shape"])
    return _mlp_raw(g, cfg), _rows(g, case["rows"], cfg.hidden_size)


def _gdn_inputs(case, seed):
    g, cfg = _gen(seed), _cfg(case["shape"])
    return _gdn_raw(g, cfg), _gdn_state(g, cfg, case["ctx"]), _rows(g, case["rows"], cfg.hidden_size)


def _attn_inputs(case, seed):
    g, cfg = _gen(seed), _cfg(case["shape"])
    return _attn_raw(g, cfg), _kv_state(g, cfg, case["ctx"]), _rows(g, case["rows"], cfg.hidden_size)


def _layer_inputs(case, seed):
    g, cfg = _gen(seed), _cfg(case["shape"])
    mixer = _gdn_raw(g, cfg) if case["linear"] else _attn_raw(g, cfg)
    hist = _gdn_state(g, cfg, case["ctx"]) if case["linear"] else _kv_state(g, cfg, case["ctx"])
    H = cfg.hidden_size
    norms = [_norm_w(g, H) for _ in range(3)]
    return mixer, _mlp_raw(g, cfg), norms, hist, _rows(g, case["rows"], H)


def _draft_inputs(case, seed):
    g, cfg = _gen(seed), _cfg(case["shape"])
    H, V = cfg.hidden_size, cfg.vocab_size
    raw = {"embed": _affine(g, V, H, gain=math.sqrt(H)), "lm_head": _affine(g, V, H, gain=2.0),
           "fc": _affine(g, H, 2 * H), "attn": _attn_raw(g, cfg), "mlp": _mlp_raw(g, cfg)}
    for n in ("norm", "norm_emb", "norm_hid", "norm_out", "ln1", "ln2"):
        raw[n] = _norm_w(g, H)
    token = int(torch.randint(0, V, (1,), generator=g, device=DEV))
    return raw, _kv_state(g, cfg, case["ctx"]), _rows(g, 1, H), token


def _accept_inputs(case, seed):
    g = _gen(seed)
    S, k, V = case["steps"], case["drafts"], case["vocab"]
    target = 3.0 * torch.randn((S, k + 1, V), generator=g, device=DEV)
    peaks = torch.randint(0, V, (S, k + 1, 2), generator=g, device=DEV)
    target.scatter_add_(2, peaks, torch.full(peaks.shape, 8.0, device=DEV))
    draft = target[:, :k] + torch.randn((S, k, V), generator=g, device=DEV)
    t = case["temperature"] or 1.0
    ids = torch.multinomial(torch.softmax(draft.reshape(S * k, V) / t, dim=-1), 1, generator=g)
    ids = ids.to(torch.int32).reshape(S, k)
    ua, us = torch.rand((S, k), generator=g, device=DEV), torch.rand(S, generator=g, device=DEV)
    if not case["draft_logits"]:
        return target.to(BF16), None, ids, ua, us
    return target, draft, ids, ua, us


def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        a, x = _linear_inputs(case, seed)
        return {"case": case, "op": _qlinear(a), "x": x}
    if kind == "mlp":
        raw, x = _mlp_inputs(case, seed)
        return {"case": case, "op": MLP(_layers_of(raw)), "x": x}
    if kind == "gdn":
        raw, (conv, state), x = _gdn_inputs(case, seed)
        cfg = _cfg(case["shape"])
        op = GatedDeltaNet(cfg, _layers_of(raw))
        return {"case": case, "op": op, "x": x, "cache": _gdn_cache(cfg, op, case["ctx"], conv, state)}
    if kind == "attn":
        raw, (k, v), x = _attn_inputs(case, seed)
        cfg = _cfg(case["shape"])
        return {"case": case, "op": Attention(cfg, _layers_of(raw)), "x": x,
                "cache": _kv_cache(cfg, case["ctx"], case["rows"], k, v)}
    if kind == "layer":
        return _prepare_layer(case, seed)
    if kind == "draft":
        return _prepare_draft(case, seed)
    if kind == "verify":
        return _prepare_verify(case, seed)
    if kind == "prefill":
        cfg = _cfg(case["shape"])
        model = random_model(cfg, seed=seed, device=DEV, max_context=MAX_CONTEXT, keep_mlx=True)
        ids = torch.randint(0, cfg.vocab_size, (1, case["rows"]), generator=_gen(seed), device=DEV, dtype=torch.int32)
        return {"case": case, "model": model, "mtp": random_mtp(model, seed=seed + 1, keep_mlx=True), "ids": ids}
    target, draft, ids, ua, us = _accept_inputs(case, seed)
    ws = kernels.spec_workspace(case["steps"], case["drafts"], case["vocab"], draft is not None, DEV, case["top_k"],
                                zeroed=False)
    return {"case": case, "target": target, "draft": draft, "ids": ids, "ua": ua, "us": us, "ws": ws}


def _prepare_layer(case, seed):
    mixer, mlp, norms, hist, x = _layer_inputs(case, seed)
    cfg = _cfg(case["shape"])
    p = {"input_layernorm": norms[0], "post_attention_layernorm": norms[1], "mlp": _layers_of(mlp)}
    if case["linear"]:
        p["linear_attn"] = _layers_of(mixer)
        layer = Layer(cfg, 0, p)
        cache = _gdn_cache(cfg, layer.mixer, case["ctx"], *hist)
    else:
        p["self_attn"] = _layers_of(mixer)
        layer = Layer(cfg, cfg.full_attention_interval - 1, p)
        cache = _kv_cache(cfg, case["ctx"], case["rows"], *hist)

    def body():
        st = NormedRows.of(x, layer.ln1, layer.eps)
        return layer.fused(x, st, cache, True, norms[2])

    graph, (h, st) = _captured(cache.counters, body)
    out = {"h": h, "u": st.u}
    if case["linear"]:
        out["state"] = cache.ssm_ring[(case["ctx"] + case["rows"]) % cache.n_slots, 0]
    else:
        out["k"], out["v"] = cache.k, cache.v
    return {"case": case, "graph": graph, "out": out, "keep": (layer, cache, x, norms)}


def _prepare_draft(case, seed):
    raw, (k, v), h, token = _draft_inputs(case, seed)
    cfg = _cfg(case["shape"])
    model = Qwen35(cfg, QEmbedding(*raw["embed"][:3]), [], raw["norm"], _qlinear(raw["lm_head"]))
    w = {n: raw[n] for n in ("norm_emb", "norm_hid", "norm_out", "ln1", "ln2")}
    w.update(fc=_qlinear(raw["fc"]), attn=_layers_of(raw["attn"]), mlp=_layers_of(raw["mlp"]))
    head = MTPHead(model, w)
    cache = _kv_cache(cfg, case["ctx"], 1, k, v)
    ids = torch.tensor([[token]], dtype=torch.int32, device=DEV)
    hid = h.view(1, 1, -1)

    def body():
        return head(hid, ids, cache, last_only=True, return_hidden=True)

    graph, (logits, hidden) = _captured(cache.counters, body)
    return {"case": case, "graph": graph, "keep": (head, cache, hid, ids),
            "out": {"logits": logits, "hidden": hidden, "k": cache.k, "v": cache.v}}


def _prepare_verify(case, seed):
    cfg, g, ctx, rows = _cfg(case["shape"]), _gen(seed), case["ctx"], case["rows"]
    model = random_model(cfg, seed=seed, device=DEV, max_context=MAX_CONTEXT, max_width=WIDTH, keep_mlx=True)
    caches = model.make_cache()
    for c in caches:
        if isinstance(c, RecurrentCache):
            c.conv_ring.copy_(_rows(g, *c.conv_ring.shape))
            c.ssm_ring[ctx % c.n_slots].normal_(0.0, 0.02, generator=g)
        else:
            c.k.normal_(generator=g)
            c.v.normal_(generator=g)
        c.offset = ctx
    caches.counters.sync()
    ids = torch.randint(0, cfg.vocab_size, (1, rows), generator=g, device=DEV, dtype=torch.int32)

    def body():
        return model(ids, caches, last_only=False, return_hidden=True, keep_prev=True)

    graph, (logits, hidden) = _captured(caches.counters, body)
    out = {"logits": logits, "hidden": hidden, "state": _new_state(caches, ctx, rows)}
    return {"case": case, "graph": graph, "out": out, "keep": (model, caches, ids)}


def _new_state(caches, ctx, rows):
    """Each layer's state after rows ctx .. ctx + rows: the DeltaNet state, or the tiles of the new keys and values."""
    new = []
    for c in caches:
        if isinstance(c, RecurrentCache):
            new.append(c.ssm_ring[(ctx + rows) % c.n_slots, 0])
        else:
            new += [c.k[:, ctx // 16:(ctx + rows + 15) // 16], c.v[:, ctx // 32:(ctx + rows + 31) // 32]]
    return new


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear" or kind == "mlp":
        return state["op"](state["x"])
    if kind == "gdn" or kind == "attn":
        cache, ctx = state["cache"], case["ctx"]
        cache.offset = ctx
        y = state["op"](state["x"], cache)
        return {"y": y, "state": cache.ssm[0]} if kind == "gdn" else {"y": y, "k": cache.k, "v": cache.v}
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    if kind == "prefill":
        model, head = state["model"], state["mtp"]
        caches = model.make_cache()
        logits, hidden = prefill(model, state["ids"], caches, head, head.make_cache())
        return {"logits": logits, "hidden": hidden, "state": _new_state(caches, 0, case["rows"])}
    n, token = kernels.spec_accept(state["target"], state["draft"], state["ids"], state["ua"], state["us"],
                                   case["temperature"], workspace=state["ws"], top_k=case["top_k"],
                                   top_p=case["top_p"])
    return {"n": n, "token": token}


# ---------------------------------------------------------------- what a pass cannot do without

def _lin(m, n, k, bits=4, group=64):
    """(bytes of the weights, flops) of one product."""
    return n * k * bits / 8 + 4 * n * k / group, 2.0 * m * n * k


def _mlp_work(cfg, m):
    H, I = cfg.hidden_size, cfg.intermediate_size
    a, b = _lin(m, 2 * I, H), _lin(m, H, I)
    return a[0] + b[0], a[1] + b[1]


def _gdn_work(cfg, m):
    H, hv, dk = cfg.hidden_size, cfg.linear_num_value_heads, cfg.linear_key_head_dim
    kd, vd = cfg.linear_num_key_heads * dk, hv * cfg.linear_value_head_dim
    a, b = _lin(m, 2 * kd + 2 * vd + 2 * hv, H), _lin(m, H, vd)
    states = 4 * vd * dk * (1 + (m if m <= WIDTH else 1))      # the state in, and each kept one out
    return a[0] + b[0] + states, a[1] + b[1] + 6.0 * m * vd * dk


def _attn_work(cfg, m, ctx):
    H, D, hq, hkv = cfg.hidden_size, cfg.head_dim, cfg.num_attention_heads, cfg.num_key_value_heads
    a, b = _lin(m, (2 * hq + 2 * hkv) * D, H), _lin(m, H, hq * D)
    kv = 2 * 2 * hkv * D * (ctx + m)
    return a[0] + b[0] + kv, a[1] + b[1] + 4.0 * hq * D * (m * ctx + m * (m + 1) / 2)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["rows"], case["n"], case["k"]
        b, f = _lin(m, n, k, case["bits"], case["group"])
        return {"bytes": b + 2 * m * (n + k), "flops": f}
    if kind == "accept":
        S, k, V = case["steps"], case["drafts"], case["vocab"]
        rows = (2 * k + 1) * 4 if case["draft_logits"] else (k + 1) * 2
        return {"bytes": S * V * rows, "flops": 0}
    cfg = _cfg(case["shape"])
    H, V = cfg.hidden_size, cfg.vocab_size
    if kind == "draft":
        parts = [_lin(1, H, 2 * H), _attn_work(cfg, 1, case["ctx"]), _mlp_work(cfg, 1), _lin(1, V, H)]
        return {"bytes": sum(p[0] for p in parts) + 2 * (2 * H + V), "flops": sum(p[1] for p in parts)}
    m = case["rows"]
    if kind == "mlp":
        b, f = _mlp_work(cfg, m)
    elif kind == "gdn":
        b, f = _gdn_work(cfg, m)
    elif kind == "attn":
        b, f = _attn_work(cfg, m, case["ctx"])
    elif kind == "layer":
        mix = _gdn_work(cfg, m) if case["linear"] else _attn_work(cfg, m, case["ctx"])
        mlp = _mlp_work(cfg, m)
        b, f = mix[0] + mlp[0], mix[1] + mlp[1]
    else:
        b, f = _lin(m if kind == "verify" else 1, V, H)
        b += 2 * (V * (m if kind == "verify" else 1))
        for i in range(cfg.num_hidden_layers):
            mix = _gdn_work(cfg, m) if cfg.is_linear(i) else _attn_work(cfg, m, case.get("ctx", 0))
            mlp = _mlp_work(cfg, m)
            b, f = b + mix[0] + mlp[0], f + mix[1] + mlp[1]
        if kind == "prefill":      # the MTP head on every pair of the prompt
            parts = [_lin(m, H, 2 * H), _attn_work(cfg, m, 0), _mlp_work(cfg, m), _lin(1, V, H)]
            b, f = b + sum(p[0] for p in parts), f + sum(p[1] for p in parts)
    return {"bytes": b + 2 * 2 * m * H, "flops": f}


def tolerance(case):
    kind = case["kind"]
    if kind == "accept":
        return "exact"
    # Measured against exact(): linear 2.2e-3, the mixers, the MLP and a layer 5e-3, a draft step 6e-3. Whole models:
    # 1.9e-3 between the folded and the separate norms, 0.8e-3 between chunks of 512 and of 300 tokens.
    return {"rel": 1e-2 if kind == "linear" else 2e-2}


# ---------------------------------------------------------------- the same in 64 bits

def _codes(w, bits):
    """uint codes [N, K] of little-endian bit-stream rows of 32-bit words."""
    words = w.to(torch.int64) & 0xFFFFFFFF
    words = torch.cat([words, words.new_zeros((words.shape[0], 1))], dim=1)
    o = torch.arange(w.shape[1] * 32 // bits, device=w.device) * bits
    wi, sh = o >> 5, o & 31
    return ((words[:, wi] | (words[:, wi + 1] << 32)) >> sh) & ((1 << bits) - 1)


def _mul64(x, a, rows=16384):
    """x W^T in 64 bits, W dequantized a block of rows at a time."""
    w, s, b, bits, group = a
    out = []
    for r in range(0, w.shape[0], rows):
        e = slice(r, r + rows)
        W = _codes(w[e], bits).double()
        W = W * s[e].double().repeat_interleave(group, dim=1) + b[e].double().repeat_interleave(group, dim=1)
        out.append(x @ W.T)
    return torch.cat(out, dim=1)


def _rms64(x, w=None, eps=1e-6):
    y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)
    return y if w is None else y * w.double()


def _silu64(x):
    return x * torch.sigmoid(x)


def _mlp64(raw, x):
    return _mul64(_silu64(_mul64(x, raw["gate_proj"])) * _mul64(x, raw["up_proj"]), raw["down_proj"])


def _gdn64(cfg, raw, hist, x):
    """The DeltaNet mixer on rows x [S, H]: (y, state after the last row)."""
    conv, state = hist[0].double(), hist[1].double()
    S, hk, hv, dk = x.shape[0], cfg.linear_num_key_heads, cfg.linear_num_value_heads, cfg.linear_key_head_dim
    kd, kw = hk * dk, cfg.linear_conv_kernel_dim
    qkv = torch.cat([conv, _mul64(x, raw["in_proj_qkv"])])
    cw = raw["conv1d"].double()
    c = _silu64(sum(qkv[j:j + S] * cw[:, j] for j in range(kw)))
    q = _rms64(c[:, :kd].reshape(S, hk, dk)) / dk
    k = _rms64(c[:, kd:2 * kd].reshape(S, hk, dk)) / math.sqrt(dk)
    v = c[:, 2 * kd:].reshape(S, hv, -1)
    q, k = q.repeat_interleave(hv // hk, dim=1), k.repeat_interleave(hv // hk, dim=1)
    a, b = _mul64(x, raw["in_proj_a"]), _mul64(x, raw["in_proj_b"])
    decay = torch.exp(-torch.exp(raw["A_log"].double()) * torch.nn.functional.softplus(a + raw["dt_bias"].double()))
    beta = torch.sigmoid(b)
    ys = []
    for t in range(S):
        state = state * decay[t][:, None, None]
        delta = (v[t] - (state @ k[t][:, :, None])[..., 0]) * beta[t][:, None]
        state = state + delta[:, :, None] * k[t][:, None, :]
        ys.append((state @ q[t][:, :, None])[..., 0])
    y = _rms64(torch.stack(ys), raw["norm"], cfg.rms_norm_eps)
    z = _mul64(x, raw["in_proj_z"])
    return _mul64(_silu64(z) * y.reshape(S, -1), raw["out_proj"]), state


def _attn64(cfg, raw, hist, x, ctx):
    """The attention mixer on rows x [S, H] at positions ctx..: (y, K cache, V cache as the kernels tile them)."""
    S, D, hq, hkv = x.shape[0], cfg.head_dim, cfg.num_attention_heads, cfg.num_key_value_heads
    qg = _mul64(x, raw["q_proj"]).reshape(S, hq, 2 * D)
    q, gate = _rms64(qg[..., :D], raw["q_norm"], cfg.rms_norm_eps), qg[..., D:]
    k = _rms64(_mul64(x, raw["k_proj"]).reshape(S, hkv, D), raw["k_norm"], cfg.rms_norm_eps)
    v = _mul64(x, raw["v_proj"]).reshape(S, hkv, D)
    half = cfg.rotary_dim // 2
    freq = cfg.rope_theta ** (-torch.arange(half, device=DEV, dtype=torch.float64) / half)
    ang = (ctx + torch.arange(S, device=DEV, dtype=torch.float64))[:, None] * freq
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def rope(t):
        lo, hi = t[..., :half], t[..., half:2 * half]
        return torch.cat([lo * cos - hi * sin, lo * sin + hi * cos, t[..., 2 * half:]], dim=-1)

    q, k = rope(q).transpose(0, 1), rope(k).transpose(0, 1)
    K = torch.cat([hist[0].double(), k], dim=1)
    V = torch.cat([hist[1].double(), v.transpose(0, 1)], dim=1)
    seen = torch.arange(ctx + S, device=DEV)[None, :] <= (ctx + torch.arange(S, device=DEV))[:, None]
    o = []
    for h in range(hq):
        s = (q[h] @ K[h * hkv // hq].T) / math.sqrt(D)
        o.append(torch.softmax(s.masked_fill(~seen, -math.inf), dim=-1) @ V[h * hkv // hq])
    o = torch.stack(o, dim=1) * torch.sigmoid(gate)
    cap = _capacity(ctx, S)
    return _mul64(o.reshape(S, hq * D), raw["o_proj"]), _tile_k(_padded(K, cap)), _tile_v(_padded(V, cap))


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        a, x = _linear_inputs(case, seed)
        return _mul64(x.double(), a)
    if kind == "mlp":
        raw, x = _mlp_inputs(case, seed)
        return _mlp64(raw, x.double())
    if kind == "gdn":
        raw, hist, x = _gdn_inputs(case, seed)
        y, state = _gdn64(_cfg(case["shape"]), raw, hist, x.double())
        return {"y": y, "state": state}
    if kind == "attn":
        raw, hist, x = _attn_inputs(case, seed)
        y, k, v = _attn64(_cfg(case["shape"]), raw, hist, x.double(), case["ctx"])
        return {"y": y, "k": k, "v": v}
    if kind == "layer":
        mixer, mlp, norms, hist, x = _layer_inputs(case, seed)
        cfg = _cfg(case["shape"])
        x = x.double()
        n = _rms64(x, norms[0], cfg.rms_norm_eps)
        if case["linear"]:
            d, state = _gdn64(cfg, mixer, hist, n)
            out = {"state": state}
        else:
            d, k, v = _attn64(cfg, mixer, hist, n, case["ctx"])
            out = {"k": k, "v": v}
        h = x + d
        h = h + _mlp64(mlp, _rms64(h, norms[1], cfg.rms_norm_eps))
        return {"h": h, "u": h * norms[2].double(), **out}
    if kind == "draft":
        raw, hist, hid, token = _draft_inputs(case, seed)
        cfg = _cfg(case["shape"])
        e = raw["embed"]
        row = torch.eye(1, device=DEV, dtype=torch.float64)
        one = tuple(t[token:token + 1] for t in e[:3])
        emb = _codes(one[0], 4).double() * one[1].double().repeat_interleave(64, dim=1) + \
            one[2].double().repeat_interleave(64, dim=1)
        eps = cfg.rms_norm_eps
        x = _mul64(torch.cat([_rms64(row @ emb, raw["norm_emb"], eps), _rms64(hid.double(), raw["norm_hid"], eps)],
                             dim=1), raw["fc"])
        d, k, v = _attn64(cfg, raw["attn"], hist, _rms64(x, raw["ln1"], eps), case["ctx"])
        h = x + d
        h = h + _mlp64(raw["mlp"], _rms64(h, raw["ln2"], eps))
        logits = _mul64(_rms64(h, raw["norm_out"], eps), raw["lm_head"])
        return {"logits": logits.view(1, 1, -1), "hidden": h.view(1, 1, -1), "k": k, "v": v}
    return None     # whole numbers by definition (accept), and whole models
