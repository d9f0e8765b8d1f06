"""The work this package is measured on: the calls a runtime makes for every
token and every prompt, through the public entry points of `spissa_amd.device`.

Kinds (each a direction of the path; head shapes and projection sizes are the
Llama 3.2 and Gemma 3 ones this repository's benchmark and tests use):

  decode    one token of `layers` layers: RoPE, attention over the cache, append
            (decode_step, or gemma_decode_step with the QK-norm), for one
            sequence or a batch of them
  prefill   a prompt or a chunk against a cache, the same three steps for many
            tokens (prefill_step, gemma_prefill_step)
  linear    a projection of resident weights (linear)
  sublayer  a layer's whole attention sublayer, norm to o projection
            (attention_sublayer)
  lm_head   the tied output table and the greedy token (lm_head)

Caches hold their rows when a pass begins and are rolled back to them by the
next pass (truncate, as a session that regenerates a turn does), so a pass can
be repeated. Weights and caches of the layers of one pass are distinct, as a
model's are: nothing is served from a cache line the layer before left behind.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from spissa_amd.device import AttentionLayer, Session
from spissa_amd.linear import DTYPE_BF16, DTYPE_F16, DTYPE_F32
from spissa_amd.rotary import KvAttentionConfig

DEV = "cuda"
EPS = 1e-6
LLAMA, GEMMA = 0, 1  # rope kinds

# hidden size, query heads, KV heads, head dim, RoPE kind, sliding window of the
# local layers, position divisor of the global layers
MODELS = {
    "llama1b": (2048, 32, 8, 64, LLAMA, 0, 1.0),
    "llama3b": (3072, 24, 8, 128, LLAMA, 0, 1.0),
    "gemma1b": (1152, 4, 1, 256, GEMMA, 512, 1.0),
    "gemma4b": (2560, 8, 4, 256, GEMMA, 1024, 8.0),
}
DTYPES = {"bf16": (DTYPE_BF16, torch.bfloat16, 2), "f16": (DTYPE_F16, torch.float16, 2),
          "f32": (DTYPE_F32, torch.float32, 4)}


def listed():
    return [
        # A short chat turn on the smallest model: 16 layers of 2 MB each, all latency.
        {"name": "decode_1b_512", "kind": "decode", "model": "llama1b", "cached": 512, "batch": 1, "layers": 16},
        # The headline: a long context, one sequence, every layer's 67 MB of keys and values read once.
        {"name": "decode_3b_8192", "kind": "decode", "model": "llama3b", "cached": 8192, "batch": 1, "layers": 28},
        # Serving: sixteen sequences of differing lengths share each launch.
        {"name": "decode_3b_batch16", "kind": "decode", "model": "llama3b", "cached": 8192, "batch": 16, "layers": 1},
        # Gemma 3's five sliding-window layers to one global layer, one KV head, a 32k context.
        {"name": "decode_gemma1b_32768", "kind": "decode", "model": "gemma1b", "cached": 32768, "batch": 1,
         "layers": 26},
        # The prompt of the headline shape.
        {"name": "prefill_3b_4096", "kind": "prefill", "model": "llama3b", "cached": 0, "tokens": 4096, "layers": 1},
        # A new turn against a long resident cache: a short chunk, five windowed layers and a global one.
        {"name": "chunk_gemma4b_128", "kind": "prefill", "model": "gemma4b", "cached": 16384, "tokens": 128,
         "layers": 6},
        # The fused q/k/v projection of a long prompt.
        {"name": "linear_prefill_4096", "kind": "linear", "tokens": 4096, "out": 5120, "in": 3072, "dtype": "bf16",
         "bias": False, "layers": 1},
        # The same projection for a decode batch, over the weights of eight layers.
        {"name": "linear_batch16", "kind": "linear", "tokens": 16, "out": 5120, "in": 3072, "dtype": "bf16",
         "bias": False, "layers": 8},
        # A checkpoint stored in binary16, a ragged chunk, with bias.
        {"name": "linear_f16_333", "kind": "linear", "tokens": 333, "out": 2048, "in": 2048, "dtype": "f16",
         "bias": True, "layers": 1},
        # One generated token through the attention sublayers of eight layers.
        {"name": "sublayer_decode_3b", "kind": "sublayer", "model": "llama3b", "cached": 2049, "tokens": 1,
         "layers": 8},
        # A ragged prompt through six Gemma sublayers (five local, one global).
        {"name": "sublayer_prefill_gemma1b", "kind": "sublayer", "model": "gemma1b", "cached": 0, "tokens": 1500,
         "layers": 6},
        # The tied table and the greedy choice after the last layer of every generated token.
        {"name": "lm_head_3b", "kind": "lm_head", "vocab": 128256, "hidden": 3072, "dtype": "bf16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "linear", "linear", "sublayer", "sublayer", "lm_head"])
    model = rng.choice(sorted(MODELS))
    hq, hkv, d = MODELS[model][1:4]
    if kind == "decode":
        batch = rng.choice([1, 1, 2, _log(rng, 3, 16)])
        layers = rng.randint(1, max(1, 24 // batch))
        most = 1.9e9 / (layers * batch * hkv * d * 8)  # the largest listed pass reads about 1.9 GB
        return {"kind": kind, "model": model, "cached": _log(rng, 2, min(32768, most)), "batch": batch, "layers": layers}
    if kind == "prefill":
        cached = rng.choice([0, _log(rng, 2, 16384)])
        layers = rng.randint(1, 6)
        most = 100e9 / (4 * d * hq * layers)  # unmasked pairs of the largest listed prompt
        most = int(math.sqrt(cached * cached + 2 * most)) - cached
        return {"kind": kind, "model": model, "cached": cached, "tokens": _log(rng, 2, max(3, min(4096, most))),
                "layers": layers}
    if kind == "linear":
        dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
        hidden = MODELS[model][0]
        out, inner = rng.choice([((hq + 2 * hkv) * d, hidden), (hkv * d, hidden), (hidden, hq * d),
                                 (_log(rng, 33, 6000), 8 * rng.randint(16, 400))])
        most = 4096 if dtype == "bf16" else min(4096, int(1.3e9 / (out * inner)))
        tokens = _log(rng, 1, max(2, most))
        layers = rng.randint(1, 8) if tokens <= 64 and dtype == "bf16" else 1
        return {"kind": kind, "tokens": tokens, "out": out, "in": inner, "dtype": dtype, "bias": rng.random() < 0.5,
                "layers": layers}
    if kind == "sublayer":
        tokens = rng.choice([1, _log(rng, 2, 2048)])
        return {"kind": kind, "model": model, "cached": rng.choice([0, _log(rng, 2, 8192)]), "tokens": tokens,
                "layers": rng.randint(1, 8 if tokens == 1 else 4)}
    dtype = rng.choice(["bf16", "bf16", "f32"])
    hidden = MODELS[model][0]
    vocab = _log(rng, 8000, min(262144, 788e6 / (hidden * DTYPES[dtype][2])))
    return {"kind": "lm_head", "vocab": vocab, "hidden": hidden, "dtype": dtype}


# ---------------------------------------------------------------------------
# inputs and state


class _Rows:
    """Rows of a cache for torch.as_tensor, whose tensor holds this object and so the cache's memory."""

    def __init__(self, cache, ptr, shape):
        self.cache = cache
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": tuple(shape), "typestr": "<f4",
                                         "strides": None, "version": 3}


_sessions = []


def _session():
    """A program's one session, on a stream of its own."""
    if not _sessions:
        stream = torch.cuda.Stream()
        _sessions.append((Session(0, stream=stream), stream))
    return _sessions[0][0]


class _Draws:
    """Seeded device tensors."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEV)
        self.gen.manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0, dtype=torch.float32):
        return (torch.randn(*shape, generator=self.gen, device=DEV) * std + mean).to(dtype)


def _is_global(model, layer):
    return MODELS[model][4] == LLAMA or (layer + 1) % 6 == 0


def _base(model, layer):
    if MODELS[model][4] == LLAMA:
        return 500000.0, 1.0
    return (1000000.0, MODELS[model][6]) if _is_global(model, layer) else (10000.0, 1.0)


def _lens(case):
    """Cached tokens of each sequence: a batch's lengths spread down to a quarter of the longest, odd ones among them."""
    p, b = case["cached"], case.get("batch", 1)
    return [max(1, p - (3 * p * i) // (4 * b)) for i in range(b)] if b > 1 else [p]


def _inputs(case, seed):
    """Every input tensor of a case, the same for prepare() and exact()."""
    r = _Draws(seed)
    kind, layers = case["kind"], case.get("layers", 1)
    if kind == "lm_head":
        dtype = DTYPES[case["dtype"]][1]
        return {"table": r.normal(case["vocab"], case["hidden"], std=0.02, dtype=dtype),
                "hidden": r.normal(case["hidden"])}
    if kind == "linear":
        m, n, k, dtype = case["tokens"], case["out"], case["in"], DTYPES[case["dtype"]][1]
        return {"w": [r.normal(n, k, std=0.02, dtype=dtype) for _ in range(layers)], "x": r.normal(layers, m, k),
                "bias": r.normal(layers, n) if case["bias"] else None}
    hidden, hq, hkv, d, rope = MODELS[case["model"]][:5]
    lens, s = _lens(case), case.get("tokens", 1)
    b = len(lens)
    got = {"past_k": [[r.normal(p, hkv, d) for p in lens] for _ in range(layers)],
           "past_v": [[r.normal(p, hkv, d) for p in lens] for _ in range(layers)]}
    if rope == GEMMA:
        got["q_norm"], got["k_norm"] = r.normal(layers, d, std=0.1, mean=1.0), r.normal(layers, d, std=0.1, mean=1.0)
    if kind == "sublayer":
        shapes = {"q": (hq * d, hidden), "k": (hkv * d, hidden), "v": (hkv * d, hidden), "o": (hidden, hq * d)}
        got["w"] = [{t: r.normal(*shape, std=0.02, dtype=torch.bfloat16) for t, shape in shapes.items()}
                    for _ in range(layers)]
        got["x"] = r.normal(layers, s, hidden)
        got["in_norm"] = r.normal(layers, hidden, std=0.1, mean=1.0)
        got["post_norm"] = r.normal(layers, hidden, std=0.1, mean=1.0) if rope == GEMMA else None
    else:  # b sequences of one token, or one sequence of s
        got["q"], got["k"], got["v"] = (r.normal(layers, b * s, h, d) for h in (hq, hkv, hkv))
    return got


def _caches(ses, case, inp):
    """caches[layer][sequence] holding their past rows, as a prompt's prefill leaves
    them (with the bf16 operands that the next prefill reads), and tensors over the
    rows the pass appends."""
    hq, hkv, d = MODELS[case["model"]][1:4]
    lens, s, w = _lens(case), case.get("tokens", 1), MODELS[case["model"]][2] * MODELS[case["model"]][3]
    caches, appended = [], []
    q, out = torch.ones(2, 2, hq, d, device=DEV).unbind()
    torch.cuda.synchronize()
    for layer in range(case["layers"]):
        row = []
        for i, p in enumerate(lens):
            c = ses.kv_cache(hkv, d, p + s + 64)
            if p:
                ses.append(c, inp["past_k"][layer][i], inp["past_v"][layer][i], p)
            if p >= 2:
                ses.attention_cached(q, c, KvAttentionConfig(2, hq, hkv, d, True), out)
            appended += [torch.as_tensor(_Rows(c, ptr + p * w * 4, (s, hkv, d)), device=DEV)
                         for ptr in (c.device_keys_ptr(), c.device_values_ptr())]
            row.append(c)
        caches.append(row)
    torch.cuda.synchronize()
    return caches, appended


def _tables(ses, case):
    kind, d = MODELS[case["model"]][4], MODELS[case["model"]][3]
    n = max(_lens(case)) + case.get("tokens", 1) + 64
    made = {}
    for layer in range(case["layers"]):
        key = _base(case["model"], layer)
        if key not in made:
            made[key] = ses.rope_table(kind, d, key[0], key[1], None, max_positions=n)
    return [made[_base(case["model"], layer)] for layer in range(case["layers"])]


def prepare(case, seed):
    ses = _session()
    inp = _inputs(case, seed)
    torch.cuda.synchronize()
    kind = case["kind"]
    st = {"case": case, "session": ses}
    if kind == "lm_head":
        st["table"] = ses.linear_weight(inp["table"], DTYPES[case["dtype"]][0], case["vocab"], case["hidden"])
        st["hidden"] = inp["hidden"]
        st["outputs"] = (torch.zeros(case["vocab"], device=DEV), torch.zeros(1, dtype=torch.int32, device=DEV))
    elif kind == "linear":
        st["w"] = [ses.linear_weight(w, DTYPES[case["dtype"]][0], case["out"], case["in"]) for w in inp["w"]]
        st["x"], st["bias"] = inp["x"], inp["bias"]
        st["outputs"] = torch.zeros(case["layers"], case["tokens"], case["out"], device=DEV)
    else:
        hidden, hq, hkv, d, rope, window, _ = MODELS[case["model"]]
        layers, b, s = case["layers"], len(_lens(case)), case.get("tokens", 1)
        st["caches"], appended = _caches(ses, case, inp)
        st["tables"], st["lens"] = _tables(ses, case), _lens(case)
        wins = [0 if _is_global(case["model"], layer) else window for layer in range(layers)]
        if kind == "sublayer":
            st["x"], out = inp["x"], torch.zeros(layers, s, hidden, device=DEV)
            st["layers"] = []
            for layer in range(layers):
                w = {t: ses.linear_weight(m, DTYPE_BF16, *m.shape) for t, m in inp["w"][layer].items()}
                pick = lambda t: inp[t][layer] if inp.get(t) is not None else None  # noqa: E731
                st["layers"].append(AttentionLayer(
                    hidden, hq, hkv, d, w["q"], w["k"], w["v"], w["o"], pick("in_norm"), pick("q_norm"),
                    pick("k_norm"), pick("post_norm"), EPS, st["tables"][layer], 1.0, True, wins[layer]))
        else:
            st["q"], st["k"], st["v"] = inp["q"], inp["k"], inp["v"]
            st["q_norm"], st["k_norm"] = inp.get("q_norm"), inp.get("k_norm")
            st["cfg"] = [KvAttentionConfig(s, hq, hkv, d, True, w) for w in wins]
            out = torch.zeros(layers, b * s, hq, d, device=DEV)
        st["outputs"] = (out, appended)
    torch.cuda.synchronize()
    return st


def run(state):
    case, ses = state["case"], state["session"]
    kind = case["kind"]
    if kind == "lm_head":
        logits, token = state["outputs"]
        ses.lm_head(state["table"], state["hidden"], logits, token)
    elif kind == "linear":
        x, bias, out = state["x"], state["bias"], state["outputs"]
        for i, w in enumerate(state["w"]):
            ses.linear(w, x[i], None if bias is None else bias[i], case["tokens"], out[i])
    else:
        out = state["outputs"][0]
        for row in state["caches"]:
            for c, p in zip(row, state["lens"]):
                c.truncate(p)
        if kind == "sublayer":
            x = state["x"]
            for i, layer in enumerate(state["layers"]):
                ses.attention_sublayer(layer, x[i], case["tokens"], state["caches"][i][0], out[i])
        else:
            q, k, v, cfg, tables = state["q"], state["k"], state["v"], state["cfg"], state["tables"]
            qn, kn = state["q_norm"], state["k_norm"]
            for i, row in enumerate(state["caches"]):
                if kind == "decode" and qn is None:
                    ses.decode_step(tables[i], q[i], k[i], v[i], row, cfg[i], out[i])
                elif kind == "decode":
                    ses.gemma_decode_step(tables[i], q[i], k[i], v[i], row, cfg[i], qn[i], kn[i], EPS, 1.0, out[i])
                elif qn is None:
                    ses.prefill_step(tables[i], q[i], k[i], v[i], row[0], cfg[i], out[i])
                else:
                    ses.gemma_prefill_step(tables[i], q[i], k[i], v[i], row[0], cfg[i], qn[i], kn[i], EPS, 1.0, out[i])
    return state["outputs"]


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how closely another implementation agrees


def _pairs(p, s, window):
    """Unmasked (query, key) pairs of s causal queries after p cached rows."""
    seen = np.arange(p + 1, p + s + 1)
    return int((np.minimum(seen, window) if window else seen).sum())


def _attention_work(case, layer):
    """K/V rows read and written, flops of one layer's attention (q and out not counted)."""
    hq, hkv, d, _, window, _ = MODELS[case["model"]][1:]
    s, w = case.get("tokens", 1), 0 if _is_global(case["model"], layer) else window
    size = flops = 0
    for p in _lens(case):
        cached = min(p, w - 1) if w and s == 1 else min(p, w + s) if w else p
        # cached rows: f32 for a decode, their bf16 copies for a prefill; new rows read and appended in f32
        size += 2 * hkv * d * (cached * (4 if s == 1 else 2) + s * 8)
        flops += 4 * d * hq * _pairs(p, s, w)
    return size, flops


def work(case):
    kind, layers = case["kind"], case.get("layers", 1)
    if kind == "lm_head":
        v, h = case["vocab"], case["hidden"]
        return {"bytes": v * h * DTYPES[case["dtype"]][2] + 4 * (v + h), "flops": 2 * v * h}
    if kind == "linear":
        m, n, k = case["tokens"], case["out"], case["in"]
        return {"bytes": layers * (n * k * DTYPES[case["dtype"]][2] + 4 * m * (n + k)), "flops": layers * 2 * m * n * k}
    hidden, hq, hkv, d = MODELS[case["model"]][:4]
    rows = case.get("tokens", 1) * len(_lens(case))
    size = flops = 0
    for layer in range(layers):
        a = _attention_work(case, layer)
        size, flops = size + a[0], flops + a[1]
        if kind == "sublayer":
            weights = hidden * d * (2 * hq + 2 * hkv)
            size += 2 * weights + 8 * rows * hidden - 8 * rows * hkv * d  # x in, out; new k and v only written
            flops += 2 * rows * weights
        else:
            size += 8 * rows * hq * d
    return {"bytes": size, "flops": flops}


def tolerance(case):
    """About four times the largest distance from exact() over the ranges of draw()."""
    kind = case["kind"]
    if kind == "linear" or (kind == "sublayer" and case["tokens"] == 1):
        return {"rel": 1e-5, "max": 2e-4}  # f32 activations, as two bf16 halves against 16-bit weights: 2.5e-6
    if kind in ("lm_head", "decode"):
        return {"rel": 2e-6, "max": 5e-5}  # f32 products and sums: 2e-7 to 4e-7
    return {"rel": 1.3e-2, "max": 2e-1}  # bf16 queries, keys, values and probabilities: 3.3e-3


# ---------------------------------------------------------------------------
# the same in 64 bits


def _rotate(x, model, layer, first):
    """rotate-half of x [rows, heads, d] (f64); the angles are single precision, as the models define them."""
    base, divisor = _base(model, layer)
    d = x.shape[-1]
    inv = np.array([np.float32(1) / np.float32(math.pow(base, float(np.float32(2 * p) / np.float32(d))))
                    for p in range(d // 2)], dtype=np.float32)
    pos = np.arange(first, first + x.shape[0], dtype=np.float32) / np.float32(divisor)
    ang = torch.from_numpy(pos[:, None] * inv[None, :]).to(DEV).double()[:, None, :]
    a, b = x[..., :d // 2], x[..., d // 2:]
    return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], -1)


def _rms(x, w):
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w.double()


def _attend(q, keys, values, window):
    """q [s, hq, d] over keys [n, hkv, d], the last s of which are the queries' own."""
    s, hq, d = q.shape
    n, hkv = keys.shape[:2]
    at = torch.arange(n - s, n, device=DEV)[:, None]
    key = torch.arange(n, device=DEV)[None, :]
    hidden = (key > at) | ((key <= at - window) if window else False)
    out = torch.empty(s, hq, d, dtype=torch.float64, device=DEV)
    for h in range(hq):
        k, v = (t[:, h // (hq // hkv)].contiguous() for t in (keys, values))
        sc = (q[:, h].contiguous() @ k.t()) / math.sqrt(d)
        out[:, h] = torch.softmax(sc.masked_fill(hidden, -math.inf), -1) @ v
    return out


def exact(case, seed):
    inp = _inputs(case, seed)
    kind, layers = case["kind"], case.get("layers", 1)
    if kind == "lm_head":
        logits = torch.cat([part.double() @ inp["hidden"].double() for part in inp["table"].split(16384)])
        return logits, logits.argmax().reshape(1).to(torch.int32)
    if kind == "linear":
        return torch.stack([inp["x"][i].double() @ inp["w"][i].double().t() +
                            (0 if inp["bias"] is None else inp["bias"][i].double()) for i in range(layers)])
    model = case["model"]
    hidden, hq, hkv, d, rope, window, _ = MODELS[model]
    lens, s = _lens(case), case.get("tokens", 1)
    outs, appended = [], []
    for layer in range(layers):
        if kind == "sublayer":
            w = {t: m.double() for t, m in inp["w"][layer].items()}
            x = _rms(inp["x"][layer].double(), inp["in_norm"][layer])
            q, k, v = ((x @ w[t].t()).reshape(s, h, d) for t, h in (("q", hq), ("k", hkv), ("v", hkv)))
        else:
            q, k, v = (inp[t][layer].double() for t in ("q", "k", "v"))
        if rope == GEMMA:
            q, k = _rms(q, inp["q_norm"][layer]), _rms(k, inp["k_norm"][layer])
        att = []
        for i, p in enumerate(lens):
            rows = slice(i * s, (i + 1) * s)
            qr, kr, vr = _rotate(q[rows], model, layer, p), _rotate(k[rows], model, layer, p), v[rows]
            keys = torch.cat([inp["past_k"][layer][i].double(), kr])
            values = torch.cat([inp["past_v"][layer][i].double(), vr])
            att.append(_attend(qr, keys, values, 0 if _is_global(model, layer) else window))
            appended += [kr, vr]
        out = torch.cat(att)
        if kind == "sublayer":
            out = out.reshape(s, hq * d) @ w["o"].t()
            out = _rms(out, inp["post_norm"][layer]) if rope == GEMMA else out
        outs.append(out)
    return torch.stack(outs), appended
