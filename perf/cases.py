"""The workloads that this library's speed is judged by.

Each case is one call sequence of the library's public entry points on
resident weights, at a size that a program using the library meets:

* `layer`: one MoE feed-forward layer (MoeFfn.forward_dev, or
  forward_norm_residual_dev with the norm and the residual), from a single
  decoded token to a prompt, in the benchmark shapes of
  leafcutterllm_amd/configs.py;
* `engine`: the decoder model (Model.forward): a prompt per sequence, then
  decode steps whose tokens the caller supplies;
* `matmul`, `shard`: the f32 and the shard-layout quantised matrix products
  (lcmoe_matmul_f32_dev, lcmoe_shard_matmul_dev), bit-exact by contract.

`exact` recomputes a case in float64 with torch alone, from the same weight
bytes.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import leafcutterllm_amd as L
from leafcutterllm_amd import configs
from leafcutterllm_amd._lib import check

DEV = "cuda"
SHAPES = {"q8": 1, "mixtral": 2, "qwen": 3, "deepseek": 4, "e2e": 5}
# most tokens per call: the shapes' benchmark batches, and a prompt for the
# two whose experts a prompt loads heavily
MOST_T = {"q8": 64, "mixtral": 1024, "qwen": 2048, "deepseek": 256, "e2e": 512}
ENGINE_LAYERS = 4  # of the 24-layer model's shape: each layer is alike
ROPE_ABSOLUTE = 1


def _layer(name, shape, T, act="f16", residual=False):
    return {"name": name, "kind": "layer", "shape": shape, "T": T, "act": act,
            "residual": residual}


def listed():
    return [
        # one decoded token of a small Q8_0 layer: launches and latency
        _layer("q8-1", "q8", 1),
        # one decoded token of a Mixtral-8x7B layer: two experts' weights
        _layer("mixtral-1", "mixtral", 1),
        # a handful of sequences decoded together: nearly every expert is read
        _layer("mixtral-7", "mixtral", 7),
        # the largest decode batch of the headline workload
        _layer("mixtral-64", "mixtral", 64),
        # a prompt through the same layer: hundreds of tokens per expert
        _layer("mixtral-1000", "mixtral", 1000),
        # a prompt through a fine-grained layer whose routing is skewed
        _layer("qwen-1801", "qwen", 1801),
        # one decoded token of a DeepSeek-V3 layer: 9 of 257 experts
        _layer("deepseek-1", "deepseek", 1),
        # a serving batch of it: a few tokens for each of 140 experts
        _layer("deepseek-150", "deepseek", 150),
        # the FFN half of a decoder layer in a batch of 16 sequences, as the
        # decoder model runs it (norm and residual fused, two f16 per activation)
        _layer("e2e-16-residual", "e2e", 16, "f16x2", True),
        # a few chats: short prompts, then decode steps
        {"name": "engine-chat", "kind": "engine", "B": 9, "P": 37, "N": 12},
        # one long prompt until its first logits
        {"name": "engine-prompt", "kind": "engine", "B": 1, "P": 500, "N": 0},
        # a shard engine's Q8_0 product for a few rows
        {"name": "shard-q8-3", "kind": "shard", "type": "q8", "m": 3, "k": 4096, "n": 14336},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)) )))))


def draw(rng):
    kind = rng.choices(["layer", "engine", "matmul", "shard"], [14, 3, 1, 2])[0]
    if kind == "layer":
        shape = rng.choices(list(SHAPES), [3, 5, 4, 3, 4])[0]
        c = _layer("", shape, _log_int(rng, 1, MOST_T[shape]),
                   "f16x2" if rng.random() < 0.25 else "f16", rng.random() < 0.3)
    elif kind == "engine":
        c = {"kind": "engine", "B": _log_int(rng, 1, 16), "P": 0, "N": rng.randint(0, 12)}
        c["P"] = _log_int(rng, 1, 512 // c["B"])
    else:
        c = {"kind": kind, "m": _log_int(rng, 1, 32), "k": 32 * _log_int(rng, 8, 128),
             "n": 32 * _log_int(rng, 8, 448)}
        if kind == "matmul":
            c["n"] = max(1, min(c["n"], 4096) - rng.choice([0, 0, 1, 6, 20]))
            c["k"] -= rng.choice([0, 0, 3, 17])
        else:
            c["type"] = rng.choice(["q8", "q4"])
    c.pop("name", None)
    return c


# ---- inputs ------------------------------------------------------------------

_stream = None


def _the_stream():
    """The one stream that a program of layers runs on."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


def _normal(seed, index, std, *shape):
    n = int(np.prod(shape))
    return configs.synth_normal(seed, index, std, n).reshape(shape)


POOL = 16381  # a prime number of blocks: no row of a matrix repeats another


@functools.lru_cache(maxsize=4)
def _pool(qtype, seed):
    bs = 32 if qtype == L.TYPE_Q8_0 else 256
    return configs.quantize(qtype, configs.synth_normal(seed, 77 + qtype, 0.02, POOL * bs))


def _bytes(qtype, seed, index, count):
    """`count` weights of N(0, 0.02) as quantised blocks: a pool of blocks,
    repeated from a place that depends on the matrix."""
    pool = _pool(qtype, seed)
    out = np.empty(configs.tensor_size(qtype, count), np.uint8)
    at, off = 0, index * 6007 % POOL * (pool.size // POOL)
    while at < out.size:
        n = min(out.size - at, pool.size - off)
        out[at:at + n] = pool[off:off + n]
        at, off = at + n, 0
    return out


def _stack(qtype, seed, index, rows, cols, n):
    return np.concatenate([_bytes(qtype, seed, index + e, rows * cols) for e in range(n)])


def _weights(cfg, seed, first=0):
    """A layer's weights as lcmoe_create takes them."""
    d, F, E, S = cfg.d_model, cfg.d_ff, cfg.n_expert, cfg.n_shared
    w = {"router": _normal(seed, first + 1, 0.02, d, E), "bias": None,
         "gate": _stack(cfg.qtype_gate, seed, first + 1000, F, d, E),
         "up": _stack(cfg.qtype_gate, seed, first + 2000, F, d, E),
         "down": _stack(cfg.qtype_down, seed, first + 3000, d, F, E)}
    if cfg.bias == "plus2_first8":
        w["bias"] = np.where(np.arange(E) < 8, 2.0, 0.0).astype(np.float32)
    elif cfg.bias == "normal0.1":
        w["bias"] = _normal(seed, first + 2, 0.1, E)
    if S:
        FS = cfg.d_ff_shared
        w["gate_sh"] = _stack(cfg.qtype_gate, seed, first + 4000, FS, d, S)
        w["up_sh"] = _stack(cfg.qtype_gate, seed, first + 5000, FS, d, S)
        w["down_sh"] = _stack(cfg.qtype_down, seed, first + 6000, d, FS, S)
    return w


def _x(seed, *shape):
    g = torch.Generator("cpu").manual_seed(seed)
    return torch.randn(*shape, generator=g, dtype=torch.float32)


def _layer_x(case, seed, d):
    """A layer's input: N(0,1); before the norm, of the size of the layer's
    output, so that neither half of the sum hides the other's error."""
    return _x(seed, case["T"], d) * (0.1 if case["residual"] else 1.0)


def _norm_weight(seed, index, d):
    return 1.0 + _normal(seed, 9000 + index, 0.02, d)


def _model_weights(mc, seed):
    d, hd, V = mc.d_model, mc.n_head * mc.head_dim, mc.vocab
    kvd = mc.n_kv_head * mc.head_dim
    qt = mc.attn_type
    layers = []
    for l in range(ENGINE_LAYERS):
        b = 20000 * (l + 1)
        layers.append({"attn_norm": _norm_weight(seed, 2 * l, d),
                       "ffn_norm": _norm_weight(seed, 2 * l + 1, d),
                       "attn_q": _bytes(qt, seed, b + 1, hd * d),
                       "attn_k": _bytes(qt, seed, b + 2, kvd * d),
                       "attn_v": _bytes(qt, seed, b + 3, kvd * d),
                       "attn_o": _bytes(qt, seed, b + 4, d * hd),
                       "moe": _weights(mc.layer, seed, b)})
    return {"token_embd": _bytes(qt, seed, 11, V * d), "output": _bytes(qt, seed, 12, V * d),
            "output_norm": _norm_weight(seed, 500, d), "layers": layers}


def _tokens(case, seed, vocab):
    rng = np.random.default_rng(seed)
    return rng.integers(0, vocab, (case["B"], case["P"] + case["N"])).astype(np.int32)


def _shard_bytes(case, seed):
    """[k, n] weights in 32-wide blocks along n: an f16 scale, then codes."""
    rng = np.random.default_rng(seed)
    k, nb = case["k"], case["n"] // 32
    q8 = case["type"] == "q8"
    if q8:  # the reference's encoder is GGUF's Q8_0
        return configs.quantize(L.TYPE_Q8_0, _normal(seed, 5, 0.02, k * nb * 32))
    out = np.empty((k * nb, 18), np.uint8)
    out[:, :2] = np.abs(rng.normal(0.006, 0.001, k * nb)).astype(np.float16).view(np.uint8).reshape(-1, 2)
    out[:, 2:] = rng.integers(0, 256, (k * nb, 16), dtype=np.uint8)
    return out.reshape(-1)


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "stream": _the_stream()}
    if kind == "layer":
        cfg = L.CONFIGS[SHAPES[case["shape"]]]
        T, d = case["T"], cfg.d_model
        m = L.MoeFfn(cfg.desc(T), _weights(cfg, seed))
        m.set_act_precision(L.ACT_F16X2 if case["act"] == "f16x2" else L.ACT_F16)
        if case["residual"]:
            m.set_norm(_norm_weight(seed, 0, d))
        s.update(moe=m, x=_layer_x(case, seed, d).to(DEV), y=torch.empty(T, d, device=DEV))
    elif kind == "engine":
        mc = L.MODEL_CONFIGS[5]
        desc = mc.desc(case["B"], case["P"], case["P"] + case["N"], ROPE_ABSOLUTE, ENGINE_LAYERS)
        s["model"] = L.Model(desc, _model_weights(mc, seed))
        t = _tokens(case, seed, mc.vocab)
        s["prompt"] = np.ascontiguousarray(t[:, :case["P"]])
        s["next"] = [np.ascontiguousarray(t[:, i:i + 1]) for i in range(case["P"], t.shape[1])]
    else:
        m, k, n = case["m"], case["k"], case["n"]
        s["a"] = _x(seed, m, k).to(DEV)
        if kind == "matmul":
            s["b"] = (_x(seed + 1000003, k, n) * 0.02).to(DEV)
        else:
            s["b"] = torch.from_numpy(_shard_bytes(case, seed)).to(DEV)
        s["c"] = torch.empty(m, n, device=DEV)
    torch.cuda.synchronize()
    return s


def run(s):
    case = s["case"]
    kind, st = case["kind"], s["stream"].cuda_stream
    if kind == "layer":
        call = s["moe"].forward_norm_residual_dev if case["residual"] else s["moe"].forward_dev
        call(s["x"].data_ptr(), case["T"], s["y"].data_ptr(), st)
        return s["y"]
    if kind == "engine":
        s["model"].reset()
        logits = [s["model"].forward(s["prompt"])]
        for t in s["next"]:
            logits.append(s["model"].forward(t))
        return logits
    m, k, n = case["m"], case["k"], case["n"]
    a, b, c = s["a"].data_ptr(), s["b"].data_ptr(), s["c"].data_ptr()
    if kind == "matmul":
        check(L.lib().lcmoe_matmul_f32_dev(a, b, c, m, k, n, st), "lcmoe_matmul_f32_dev")
    else:
        qt = L.TYPE_Q8_0 if case["type"] == "q8" else L.TYPE_Q4_0
        check(L.lib().lcmoe_shard_matmul_dev(qt, a, b, c, m, k, n, st), "lcmoe_shard_matmul_dev")
    return s["c"]


# ---- what a pass cannot do without -------------------------------------------

# experts that T tokens touch, averaged over seeds, where the bias makes them
# fewer than uniform routing would: at T = 4^0, 4^1, ...
TOUCHED = {"qwen-moe-prefill-q4_k": [4.0, 9.2, 15.6, 32.6, 56.1, 60.0, 60.0],
           "deepseek-v3-q4_k-q6_k": [8.0, 27.1, 67.4, 108.0, 136.7, 150.0, 150.0]}


def _touched(cfg, T):
    if cfg.name in TOUCHED:
        return float(np.interp(math.log(T, 4), range(7), TOUCHED[cfg.name]))
    return cfg.n_expert * (1 - (1 - cfg.n_expert_used / cfg.n_expert) ** T)


def _layer_work(cfg, T, residual=False):
    d = cfg.d_model
    b = _touched(cfg, T) * cfg.expert_bytes() + 4 * d * cfg.n_expert + 8 * T * d
    if cfg.n_shared:
        b += cfg.n_shared * cfg.shared_bytes()
    f = 6.0 * d * T * (cfg.d_ff * cfg.n_expert_used + cfg.d_ff_shared * cfg.n_shared)
    return b + (4 * d if residual else 0), f + 2.0 * T * d * cfg.n_expert


def work(case):
    kind = case["kind"]
    if kind == "layer":
        b, f = _layer_work(L.CONFIGS[SHAPES[case["shape"]]], case["T"], case["residual"])
        return {"bytes": b, "flops": f}
    if kind == "engine":
        mc, B, P, N = L.MODEL_CONFIGS[5], case["B"], case["P"], case["N"]
        d, hd, V = mc.d_model, mc.n_head * mc.head_dim, mc.vocab
        attn = 4 * configs.tensor_size(mc.attn_type, d * hd)
        head = configs.tensor_size(mc.attn_type, V * d)
        b = f = 0.0
        # the prompts, one sequence a call (together where they are one token), then the steps
        calls = [(1, P)] * B if P > 1 else [(B, 1)]
        for nseq, T in calls + [(B, 1)] * N:
            lb, lf = _layer_work(mc.layer, nseq * T, True)
            b += ENGINE_LAYERS * (attn + lb + 2 * 2 * nseq * (P + N / 2) * hd) + head + 4 * nseq * V
            f += ENGINE_LAYERS * (8.0 * nseq * T * d * hd + lf + 4.0 * nseq * T * (P + T) / 2 * hd)
            f += 2.0 * nseq * d * V
        return {"bytes": b, "flops": f}
    m, k, n = case["m"], case["k"], case["n"]
    wb = 4.0 * k * n if kind == "matmul" else k * n / 32 * (34 if case["type"] == "q8" else 18)
    return {"bytes": wb + 4.0 * m * (k + n), "flops": 2.0 * m * k * n}


def tolerance(case):
    kind = case["kind"]
    if kind == "layer":
        cfg = L.CONFIGS[SHAPES[case["shape"]]]
        T = case["T"]
        # up to three tokens (up to a token per expert for Q8_0): exact products
        # of 15-bit activations, 9e-5 against float64
        few = T * cfg.n_expert_used <= cfg.n_expert and (T < 4 or case["shape"] == "q8")
        if few or (case["act"] == "f16x2" and case["shape"] == "q8"):
            return {"rel": 4e-4}
        # one f16 per activation, 3.6e-4 against float64; two, 0.6e-6 to 1.7e-6
        return {"rel": 7e-6 if case["act"] == "f16x2" else 1.4e-3}
    if kind == "engine":
        # four layers of one-token calls at 15-bit activations (9e-5 a layer)
        # or of two f16 each, on a cache in f16: up to 2.2e-4 against float64
        return {"rel": 1e-3}
    return "exact"  # the order of every sum is part of the contract


# ---- float64 -----------------------------------------------------------------

def _dequant(qtype, data, rows, cols):
    """GGUF bytes -> float64 [rows, cols] on the GPU."""
    b = torch.from_numpy(np.ascontiguousarray(data)).to(DEV)

    def half(t):  # [n, 2] bytes -> [n] float64
        return t.contiguous().view(torch.float16).double().reshape(-1)

    if qtype == L.TYPE_Q8_0:
        b = b.view(-1, 34)
        v = b[:, 2:].contiguous().view(torch.int8).double() * half(b[:, :2])[:, None]
    elif qtype == L.TYPE_Q4_K:
        b = b.view(-1, 144)
        d, dm, s, q = half(b[:, :2]), half(b[:, 2:4]), b[:, 4:16].int(), b[:, 16:]
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        q = q.view(-1, 4, 32)
        q = torch.stack([q & 15, q >> 4], 2).view(-1, 8, 32).double()
        v = (d[:, None] * sc.double())[:, :, None] * q - (dm[:, None] * mn.double())[:, :, None]
    else:  # Q6_K: low nibbles, high bit pairs, int8 scales of 16, the f16 scale
        b = b.view(-1, 210)
        ql, qh = b[:, :128].view(-1, 2, 2, 32), b[:, 128:192].view(-1, 2, 32)
        sc, d = b[:, 192:208].contiguous().view(torch.int8).double(), half(b[:, 208:210])
        lo = [ql[:, :, 0] & 15, ql[:, :, 1] & 15, ql[:, :, 0] >> 4, ql[:, :, 1] >> 4]
        q = torch.stack([lo[i] | (((qh >> (2 * i)) & 3) << 4) for i in range(4)], 2)
        q = q.reshape(-1, 16, 16).double() - 32.0
        v = q * (sc * d[:, None])[:, :, None]
    return v.reshape(rows, cols)


def _chain(x, w):
    """Router logits as the routing defines them: per output one float32
    sequence of fused multiply-adds over the inputs in order (of rounded
    products in the last E % 8 columns)."""
    E8 = w.shape[1] // 8 * 8
    x, w = x.double(), w.double()
    a = torch.zeros(x.shape[0], w.shape[1], device=DEV)
    tail = torch.arange(w.shape[1], device=DEV) >= E8
    for k in range(x.shape[1]):
        p = x[:, k:k + 1] * w[k]
        if E8 < w.shape[1]:
            p = torch.where(tail, p.float().double(), p)
        a = (a.double() + p).float()
    return a


def _route(cfg, x, w):
    """(expert indices, weights) of x [T, d]: selected by the float32 logits,
    weighed in float64."""
    W = torch.from_numpy(w["router"]).to(DEV)
    c = _chain(x.float(), W)
    logits = x.double() @ W.double()
    bias = None if w["bias"] is None else torch.from_numpy(w["bias"]).to(DEV)
    K, E = cfg.n_expert_used, cfg.n_expert
    if cfg.route_kind == L.ROUTE_SIGMOID_GROUP:
        z = torch.sigmoid(c.double()).float()
        z = z if bias is None else z + bias
        g = z.view(-1, cfg.n_group, E // cfg.n_group)
        score = g.topk(2, 2).values.sum(2)
        keep = torch.zeros_like(score).scatter_(
            1, score.argsort(dim=1, descending=True, stable=True)[:, :cfg.topk_group], 1.0)
        z = torch.where(keep.bool()[:, :, None].expand_as(g).reshape(z.shape), z, -math.inf)
        idx = z.argsort(dim=1, descending=True, stable=True)[:, :K]
        v = torch.sigmoid(logits).gather(1, idx)
        return idx, v / v.sum(1, keepdim=True) * cfg.routed_scale
    z = c if bias is None else c + bias
    idx = z.argsort(dim=1, descending=True, stable=True)[:, :K]
    z = logits if bias is None else logits + bias.double()
    if cfg.route_kind == L.ROUTE_SOFTMAX_RENORM:
        p = torch.softmax(z.gather(1, idx), 1)
    else:
        p = torch.softmax(z, 1).gather(1, idx)
    return idx, p * cfg.routed_scale


def _ffn(cfg, x, w):
    """The MoE layer of x [T, d] in float64."""
    d, x = cfg.d_model, x.double()
    idx, p = _route(cfg, x, w)
    y = torch.zeros_like(x)

    def expert(sfx, F, e, xe):
        def mat(k, qt, r, c):
            n = configs.tensor_size(qt, r * c)
            return _dequant(qt, w[k + sfx][e * n:(e + 1) * n], r, c)
        g = xe @ mat("gate", cfg.qtype_gate, F, d).T
        h = g * torch.sigmoid(g) * (xe @ mat("up", cfg.qtype_gate, F, d).T)
        return h @ mat("down", cfg.qtype_down, d, F).T

    for e in torch.unique(idx).tolist():
        t, k = (idx == e).nonzero(as_tuple=True)
        y[t] += p[t, k][:, None] * expert("", cfg.d_ff, e, x[t])
    for j in range(cfg.n_shared):
        y += expert("_sh", cfg.d_ff_shared, j, x)
    return y


def _rms(x, w):
    w = torch.from_numpy(w).to(DEV).double()
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w


def _engine(case, seed):
    """Every call's logits: the tokens of a sequence in one pass, each token
    attending to those up to it, keys and values rounded to the cache's f16."""
    mc, B, P, N = L.MODEL_CONFIGS[5], case["B"], case["P"], case["N"]
    w = _model_weights(mc, seed)
    d, H, hd, V = mc.d_model, mc.n_head, mc.head_dim, mc.vocab
    tok = torch.from_numpy(_tokens(case, seed, V).astype(np.int64)).to(DEV)
    S = P + N
    x = _dequant(mc.attn_type, w["token_embd"], V, d)[tok.reshape(-1)]
    freq = 1.0 / mc.rope_theta ** (2.0 * torch.arange(hd // 2, device=DEV).double() / hd)
    ang = torch.arange(S, device=DEV).double()[:, None] * freq
    cos, sin = torch.cos(ang)[None, :, None], torch.sin(ang)[None, :, None]

    def rope(v):
        a, b = v[..., :hd // 2], v[..., hd // 2:]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)

    later = torch.ones(S, S, dtype=torch.bool, device=DEV).triu(1)
    for lw in w["layers"]:
        n = _rms(x, lw["attn_norm"])
        q, k, v = ((n @ _dequant(mc.attn_type, lw[m], H * hd, d).T).view(B, S, H, hd)
                   for m in ("attn_q", "attn_k", "attn_v"))
        q, k, v = rope(q), rope(k).half().double(), v.half().double()
        out = torch.empty(B, S, H, hd, dtype=torch.float64, device=DEV)
        for b in range(B):
            for h in range(H):
                s = (q[b, :, h] @ k[b, :, h].T.contiguous()) / math.sqrt(hd)
                out[b, :, h] = torch.softmax(s.masked_fill(later, -math.inf), 1) @ v[b, :, h]
        x = x + out.view(B * S, H * hd) @ _dequant(mc.attn_type, lw["attn_o"], d, H * hd).T
        x = x + _ffn(mc.layer, _rms(x, lw["ffn_norm"]), lw["moe"])
    head = _dequant(mc.attn_type, w["output"], V, d).T.contiguous()
    x = _rms(x, w["output_norm"]).view(B, S, d)
    return [x[:, i] @ head for i in range(P - 1, S)]


def exact(case, seed):
    kind = case["kind"]
    if kind == "layer":
        cfg = L.CONFIGS[SHAPES[case["shape"]]]
        w, x = _weights(cfg, seed), _layer_x(case, seed, cfg.d_model).to(DEV).double()
        if not case["residual"]:
            return _ffn(cfg, x, w)
        return x + _ffn(cfg, _rms(x, _norm_weight(seed, 0, cfg.d_model)), w)
    if kind == "engine":
        return _engine(case, seed)
    m, k, n = case["m"], case["k"], case["n"]
    a = _x(seed, m, k).to(DEV).double()
    if kind == "matmul":
        return a @ (_x(seed + 1000003, k, n) * 0.02).to(DEV).double()
    b = torch.from_numpy(_shard_bytes(case, seed)).to(DEV)
    b = b.view(-1, 34 if case["type"] == "q8" else 18)
    scale = b[:, :2].contiguous().view(torch.float16).double()
    if case["type"] == "q8":
        q = b[:, 2:].contiguous().view(torch.int8).double()
    else:  # element 2t the low nibble of byte t, 2t + 1 the high one
        q = torch.stack([b[:, 2:] & 15, b[:, 2:] >> 4], 2).reshape(-1, 32).double() - 8.0
    return a @ (q * scale).view(k, n)
