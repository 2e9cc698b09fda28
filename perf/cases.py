"""Performance cases: the work a program that uses this package has it do.

A case is a dict of plain values.  `listed()` are the fixed ones, `draw(rng)` makes another one of
the same ranges, `prepare` builds what a program keeps (weights on the device, filled KV caches,
recorded steps), `run` is one pass through the public entry points, `work` what that pass cannot do
without, `tolerance` how far another correct implementation may be, `exact` the results in 64 bits.

Kinds:
  decode   tokens of a running conversation: Llama2.decode_greedy at batch 1, then the logits
  prompt   a prompt: Llama2.prefill, then the logits the first token is chosen from
  turn     the next message of a chat: a short prefill behind a filled cache, then decoding
  sampled  the chat loop with temperature and top-p: Llama2.generate_sampled
  gpt2     Gpt2.generate_greedy from a prompt
  ops      a program that composes the decoder itself from the operators (GemvQuant, RmsNorm, ...)

Weights are normal as freshly initialised models have them (standard deviation 0.02, the matrices
that write to the residual stream smaller by sqrt(2 layers)), quantized to the case's format.  The
output matrix favours one successor per token, so that, as with a trained model, the arg-max
stands clear of rounding.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import wgml_amd as W
from wgml_amd import _lib
from wgml_amd.models import (GPT2_124M, LLAMA2_7B, LLAMA3_8B, TINY_LLAMA, Gpt2, Gpt2HostWeights,
                             Gpt2Params, HostMatrix, Llama2, Llama2Config, LlamaHostWeights,
                             LlamaModelType, use_more_bits)

# scheme -> format of every matrix ("q4_k_m" mixes Q4_K and Q6_K as llama.cpp does)
FORMATS = {"q8_0": _lib.Q8_0, "q4_k": _lib.Q4_K, "q6_k": _lib.Q6_K, "q4_0": _lib.Q4_0,
           "q5_k": _lib.Q5_K, "f16": _lib.F16}
SUCCESSORS = 4096  # tokens that have a favoured successor (all that a case starts from)


def _llama(name, kind, cfg, scheme, **more):
    c = {"name": name, "kind": kind, "dim": cfg.dim, "hidden": cfg.hidden_dim, "layers": cfg.n_layers,
         "heads": cfg.n_q_heads, "kv_heads": cfg.n_kv_heads, "vocab": cfg.vocab_size,
         "rope_base": cfg.rope_base_freq, "scheme": scheme, "qwen2": False, "pos": 0, "tokens": 0,
         "steps": 0, "f32_activations": False, "plain_f16": False}
    c.update(more)
    return c


def listed():
    return [
        # the smallest model: launches and latency are all there is
        _llama("tiny_q8_0_decode", "decode", TINY_LLAMA, "q8_0", pos=16, steps=48),
        # GPT-2 124M completing a text, quantized ...
        _gpt2("gpt2_q8_0_generate", GPT2_124M, "q8_0", tokens=32, steps=96),
        # ... and as an F16 file, which runs on f32 matrices
        _gpt2("gpt2_f16_generate", GPT2_124M, "f16", tokens=8, steps=16),
        # the headline: 7B shape in the common Q4_K_M mix, decoding in a short conversation
        _llama("llama7b_q4_k_m_decode", "decode", LLAMA2_7B, "q4_k_m", pos=133, steps=16),
        # long context: grouped-query widths of the 8B shape (8 of its 32 layers) at 8192 positions
        _llama("llama8b_q6_k_decode_8k", "decode", LLAMA3_8B, "q6_k", layers=8, pos=8192, steps=8),
        # 7B widths with fp32 activations, the option for exact arithmetic, at an ordinary length
        _llama("llama7b_q8_0_decode_f32", "decode", LLAMA2_7B, "q8_0", layers=8, pos=700, steps=16,
               f32_activations=True),
        # an ordinary prompt (a quarter of the 7B shape's layers), default precision
        _llama("llama7b_q4_k_m_prompt_128", "prompt", LLAMA2_7B, "q4_k_m", layers=8, tokens=128),
        # a ragged prompt behind earlier context, in the faster precision
        _llama("llama7b_q4_k_m_prompt_45_f16", "prompt", LLAMA2_7B, "q4_k_m", layers=8, pos=300,
               tokens=45, plain_f16=True),
        # a document: many runs of the prompt pass and attention over a long context
        _llama("llama8b_q8_0_prompt_1000", "prompt", LLAMA3_8B, "q8_0", layers=4, tokens=1000),
        # the next message of a chat: 21 tokens in, 24 tokens out, 600 positions behind
        _llama("mid_q4_0_turn", "turn", Llama2Config(3072, 8192, 8, 24, 8, 32000, 1024), "q4_0",
               pos=600, tokens=21, steps=24),
        # the chat loop with temperature and nucleus sampling, Qwen2 variant (biases, Neox RoPE)
        _llama("mid_q5_k_sampled", "sampled", Llama2Config(2048, 5632, 8, 16, 4, 32000, 512), "q5_k",
               qwen2=True, tokens=12, steps=20),
        # a decoder composed from the operators, as the reference's own programs are written
        _llama("mid_q4_k_ops", "ops", Llama2Config(2048, 5632, 2, 32, 8, 32000, 512), "q4_k", pos=300),
    ]


def _gpt2(name, p, scheme, tokens, steps):
    return {"name": name, "kind": "gpt2", "dim": p.n_embd, "hidden": p.ff_len, "layers": p.n_layer,
            "heads": p.n_head, "vocab": p.n_vocab, "scheme": scheme, "pos": 0, "tokens": tokens,
            "steps": steps, "f32_activations": False, "plain_f16": False}


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("decode", "decode", "prompt", "prompt", "turn", "sampled", "gpt2", "ops"))
    if kind == "gpt2":
        heads = rng.randint(4, 16)
        p = Gpt2Params(n_vocab=_log_int(rng, 5000, 50257), n_seq=1024, n_embd=64 * heads, n_head=heads,
                       n_layer=rng.randint(2, 12), ff_len=256 * heads, attn_b=192 * heads)
        scheme = rng.choice(("q8_0", "q4_0", "f16"))
        c = _gpt2("", p, scheme, _log_int(rng, 1, 60), rng.randint(8, 100 if scheme != "f16" else 16))
    else:
        scheme = rng.choice(("q8_0", "q4_k", "q6_k", "q4_k_m", "q4_0", "q5_k"))
        if scheme in ("q8_0", "q4_0"):  # rows are whole blocks of 32 elements, else of 256
            head, unit = rng.choice((32, 64, 96, 128)), 32
            dim = head * _log_int(rng, 3, 4096 // head)
        else:
            head, unit = rng.choice((64, 128)), 256
            dim = 256 * _log_int(rng, 1, 16)
        heads = dim // head
        kv = heads // rng.choice([g for g in (1, 1, 2, 4, 8) if heads % g == 0])
        hidden = unit * int(round(rng.uniform(2.0, 3.5) * dim / unit))
        cfg = Llama2Config(dim, hidden, rng.randint(1, 4), heads, kv, _log_int(rng, 5000, 50000), 0,
                           rng.choice((10000.0, 500000.0)))
        c = _llama("", kind, cfg, scheme, qwen2=rng.random() < 0.3)
        if kind == "decode":
            c.update(pos=_log_int(rng, 1, 8200), steps=rng.randint(8, 24),
                     f32_activations=rng.random() < 0.2)
        elif kind == "prompt":
            c.update(pos=rng.choice((0, _log_int(rng, 1, 2000))), tokens=_log_int(rng, 2, 1000),
                     plain_f16=rng.random() < 0.4)
        elif kind == "turn":
            c.update(pos=_log_int(rng, 8, 2000), tokens=_log_int(rng, 2, 200), steps=rng.randint(8, 32))
        elif kind == "sampled":
            c.update(tokens=rng.randint(1, 30), steps=rng.randint(4, 20))
        else:
            c.update(pos=_log_int(rng, 1, 3000))
    del c["name"]
    return c


# ---- weights ------------------------------------------------------------------------------------

def _quantize_q4_0(x):
    b = x.reshape(-1, 32)
    top = np.take_along_axis(b, np.abs(b).argmax(1)[:, None], 1)
    d = (top / -8).astype(np.float16)
    q = np.clip(np.rint(b / np.where(d == 0, 1, d).astype(np.float32)) + 8, 0, 15).astype(np.uint8)
    return np.hstack([d.view(np.uint8), q[:, :16] | (q[:, 16:] << 4)]).reshape(-1)


def _quantize_q5_k(x):
    b = x.reshape(-1, 8, 32)
    low = np.minimum(b.min(2), 0)
    scale = (b.max(2) - low) / 31
    d = (scale.max(1, keepdims=True) / 63).astype(np.float16)
    dmin = (-low.min(1, keepdims=True) / 63).astype(np.float16)
    df, mf = d.astype(np.float32), dmin.astype(np.float32)
    sc = np.clip(np.rint(scale / df), 1, 63).astype(np.uint8)
    mn = np.clip(np.rint(-low / mf), 0, 63).astype(np.uint8)
    q = np.clip(np.rint((b + (mf * mn)[..., None]) / (df * sc)[..., None]), 0, 31).astype(np.uint8)
    packed = np.zeros((len(b), 12), np.uint8)
    packed[:, 0:4] = sc[:, :4] | ((sc[:, 4:] >> 4) << 6)
    packed[:, 4:8] = mn[:, :4] | ((mn[:, 4:] >> 4) << 6)
    packed[:, 8:12] = (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)
    qs = (q[:, 0::2] & 15) | ((q[:, 1::2] & 15) << 4)
    qh = np.zeros((len(b), 32), np.uint8)
    for s in range(8):
        qh |= (q[:, s] >> 4) << s
    return np.hstack([d.view(np.uint8), dmin.view(np.uint8), packed, qh, qs.reshape(len(b), 128)]).reshape(-1)


def _quantize(qtype, x):
    x = np.ascontiguousarray(x, np.float32).reshape(-1)
    if qtype == _lib.F16:
        return x.astype(np.float16).view(np.uint8)
    if qtype == _lib.Q4_0:
        return _quantize_q4_0(x)
    if qtype == _lib.Q5_K:
        return _quantize_q5_k(x)
    return W.quantize(qtype, x)


class _Weights:
    """Matrices of one seed.  Each is a stretch, from a place of its own, of a pool of quantized
    blocks that repeats beyond its length: quick to make, and no two matrices are the same."""

    def __init__(self, seed, elements, layers):
        self.layers = layers
        self.rng = np.random.default_rng(seed)
        self.most = max(1 << 21, min(1 << 24, 1 << (elements - 1).bit_length()))
        self.seed = seed
        self.base = W.rng_normal(seed * 1009, self.most)
        self.pools = {}  # key -> (length before it repeats, values)

    def _cut(self, key, unit, n):
        length, pool = self.pools[key]
        if len(pool) < length + n:
            pool = np.resize(pool[:length], length + n)
            self.pools[key] = (length, pool)
        start = unit * int(self.rng.integers(length // unit))
        return pool[start:start + n]

    def normal(self, n, std=1.0, pool=1):
        if pool not in self.pools:  # 1: vectors and caches, 2: embedding, 3: output matrix
            self.pools[pool] = (self.most, W.rng_normal(self.seed * 1009 + pool, self.most))
        v = self._cut(pool, 1, n)
        return v * np.float32(std) if std != 1.0 else v

    def matrix(self, qtype, rows, cols, residual=False):
        key = (qtype, residual)
        if key not in self.pools:
            std = 0.02 / math.sqrt(2 * self.layers) if residual else 0.02
            n = min(self.most, 1 << 21) if qtype in (_lib.Q4_0, _lib.Q5_K) else self.most
            pool = _quantize(qtype, self.base[:n] * np.float32(std))
            self.pools[key] = (len(pool), pool)
        return HostMatrix(qtype, rows, cols, self._cut(key, _file_bytes(qtype, 256), _file_bytes(qtype, rows * cols)))

    def embedding(self, vocab, dim):
        """Of the residual stream's size (what the layers add to it grows with their number)."""
        return self.normal(vocab * dim, math.sqrt(self.layers), 2).reshape(vocab, dim)

    def output(self, qtype, embd):
        """Logits of standard deviation 2.5, and for the first SUCCESSORS tokens t the embedding of
        t mixed into row t + 1, which raises that logit by up to 24."""
        vocab, dim = embd.shape
        std = 2.5 / math.sqrt(dim)
        s = min(SUCCESSORS, vocab - 1)
        head = self.normal(s * dim, std, 3).reshape(s, dim)
        head += np.roll(embd[:s], 1, axis=0) * np.float32(24 / math.sqrt(self.layers) / dim)
        rest = vocab - s
        n = min(self.most // dim // 8 * 8 or 8, (rest + 7) // 8 * 8)
        tail = _quantize(qtype, self.normal(n * dim, std, 3))
        tail = np.resize(tail, _file_bytes(qtype, rest * dim))
        return HostMatrix(qtype, vocab, dim, np.concatenate([_quantize(qtype, head), tail]))


def _file_bytes(qtype, n):
    return 2 * n if qtype == _lib.F16 else W.quant_bytes(qtype, n)


def _format(case, name, layer=0):
    if case["scheme"] != "q4_k_m":
        return FORMATS[case["scheme"]]
    more = name in ("attn_v", "output") or (name == "ffn_down" and use_more_bits(layer, case["layers"]))
    return _lib.Q6_K if more else _lib.Q4_K


def _llama_shapes(case):
    d, h, kv = case["dim"], case["hidden"], case["dim"] // case["heads"] * case["kv_heads"]
    return {"attn_q": (d, d), "attn_k": (kv, d), "attn_v": (kv, d), "attn_output": (d, d),
            "ffn_down": (d, h), "ffn_gate": (h, d), "ffn_up": (h, d)}


def _gpt2_shapes(case):
    d, f = case["dim"], case["hidden"]
    return {"attn_w": (3 * d, d), "attn_proj_w": (d, d), "mlp_fc_w": (f, d), "mlp_proj_w": (d, f)}


def _llama_weights(case, seed, cfg):
    shapes = _llama_shapes(case)
    w = _Weights(seed, sum(r * k for r, k in shapes.values()) * case["layers"], case["layers"])
    host = LlamaHostWeights(config=cfg)
    kv = cfg.kv_dim
    for l in range(case["layers"]):
        layer = {n: w.matrix(_format(case, n, l), r, k, n in ("attn_output", "ffn_down"))
                 for n, (r, k) in shapes.items()}
        layer["attn_norm"] = 1 + w.normal(cfg.dim, 0.1)
        layer["ffn_norm"] = 1 + w.normal(cfg.dim, 0.1)
        if case["qwen2"]:
            for n, r in (("attn_q_bias", cfg.dim), ("attn_k_bias", kv), ("attn_v_bias", kv)):
                layer[n] = w.normal(r, 0.1)
        host.layers.append(layer)
    host.token_embd = w.embedding(cfg.vocab_size, cfg.dim)
    host.output = w.output(_format(case, "output"), host.token_embd)
    host.output_norm = 1 + w.normal(cfg.dim, 0.1)
    return host, w


def _gpt2_weights(case, seed, p):
    w = _Weights(seed, 12 * p.n_embd * p.n_embd * p.n_layer, p.n_layer)
    qtype = _format(case, "")
    host = Gpt2HostWeights(params=p)
    for _ in range(p.n_layer):
        layer = {n: w.matrix(qtype, r, k, n.endswith("proj_w")) for n, (r, k) in _gpt2_shapes(case).items()}
        for n, k in (("attn_b", p.attn_b), ("attn_proj_b", p.n_embd), ("mlp_fc_b", p.ff_len),
                     ("mlp_proj_b", p.n_embd), ("ln_1_b", p.n_embd), ("ln_2_b", p.n_embd)):
            layer[n] = w.normal(k, 0.02)
        for n in ("ln_1_g", "ln_2_g"):
            layer[n] = 1 + w.normal(p.n_embd, 0.1)
        host.layers.append(layer)
    host.wte = w.embedding(p.n_vocab, p.n_embd)
    host.wpe = w.normal(p.n_seq * p.n_embd, 0.1).reshape(p.n_seq, p.n_embd)
    host.lm_head = w.output(qtype, host.wte)
    host.ln_f_g, host.ln_f_b = 1 + w.normal(p.n_embd, 0.1), w.normal(p.n_embd, 0.02)
    return host


# ---- prepare and run ----------------------------------------------------------------------------

def _gpt2_params(case):
    return Gpt2Params(case["vocab"], 1024, case["dim"], case["heads"], case["layers"], case["hidden"],
                      3 * case["dim"])


def _llama_config(case):
    positions = case["pos"] + case["tokens"] + case["steps"] + 1
    return Llama2Config(case["dim"], case["hidden"], case["layers"], case["heads"], case["kv_heads"],
                        case["vocab"], max(512, (positions + 255) // 256 * 256), case["rope_base"], 1.0e-5)


def prepare(case, seed):
    gpu = W.GpuInstance(0)
    tokens = W.rng_tokens(seed + 17, max(1, case["tokens"]), min(SUCCESSORS, case["vocab"]) - 1)
    state = {"case": case, "gpu": gpu, "tokens": tokens, "seed": seed}
    if case["kind"] == "gpt2":
        p = _gpt2_params(case)
        state["model"] = Gpt2(gpu, p).load(_gpt2_weights(case, seed, p))
        state["model"].record_steps(case["tokens"] + case["steps"])
        return state
    cfg = _llama_config(case)
    host, w = _llama_weights(case, seed, cfg)
    if case["kind"] == "ops":
        return _prepare_ops(state, cfg, host, w)
    if case["f32_activations"]:
        gpu.set_tuning(gpu.TUNE_GEMV_F32_ACTIVATIONS, 1)
    if case["plain_f16"]:
        gpu.set_gemm_precision(0)
    model = Llama2(gpu, cfg, LlamaModelType.Qwen2 if case["qwen2"] else LlamaModelType.Llama).load(host)
    if case["pos"]:  # what the conversation so far has left in the cache
        for l in range(cfg.n_layers):
            for which in (0, 1):
                model.kv_upload(l, which, 0, w.normal(case["pos"] * cfg.kv_dim))
    if case["kind"] == "decode":
        model.record_steps(case["pos"], case["steps"])
    if case["kind"] == "turn":
        model.record_steps(case["pos"] + case["tokens"], case["steps"])
    state["model"] = model
    return state


def _prepare_ops(state, cfg, host, w):
    gpu, n = state["gpu"], cfg.seq_len
    vec = lambda v: W.GpuVector.init(gpu, v)  # noqa: E731
    mat = lambda m: W.GpuQuantMatrix(gpu, m.qtype, m.nrows, m.ncols, m.data)  # noqa: E731
    state["layers"] = [
        {k: mat(v) if isinstance(v, HostMatrix) else vec(v) for k, v in layer.items()}
        | {c: W.GpuMatrix.init(gpu, w.normal(n * cfg.kv_dim).reshape(n, cfg.kv_dim)) for c in ("keys", "values")}
        for layer in host.layers]
    state["embd"] = W.GpuMatrix.init(gpu, host.token_embd)
    state["output"], state["output_norm"] = mat(host.output), vec(host.output_norm)
    for name, size in (("x", cfg.dim), ("xb", cfg.dim), ("q", cfg.dim), ("att", cfg.dim), ("out", cfg.dim),
                       ("gate", cfg.hidden_dim), ("up", cfg.hidden_dim), ("logits", cfg.vocab_size)):
        state[name] = W.GpuVector.uninit(gpu, size)
    state["ops"] = (W.GemvQuant.from_device(gpu), W.RmsNorm.from_device(gpu), W.RoPE.from_device(gpu),
                    W.BatchedMultiqueryAttention.from_device(gpu), W.Silu.from_device(gpu),
                    W.OpAssign(gpu, W.OpAssignVariant.Add), W.Sampler(gpu))
    state["config"] = cfg
    return state


def _run_ops(s):
    gemv, norm, rope, attention, silu, add, sampler = s["ops"]
    cfg, case, pos = s["config"], s["case"], s["case"]["pos"]
    variant = W.RoPEVariant.Neox if case["qwen2"] else W.RoPEVariant.Original
    rms = W.RmsNormConfig(cfg.rms_norm_eps)
    rope_cfg = W.RoPEConfig(cfg.head_size, cfg.kv_dim, pos, cfg.rope_base_freq)
    params = W.BatchedMultiqueryAttentionParams(cfg.seq_len, cfg.kv_dim, cfg.n_q_heads // cfg.n_kv_heads,
                                                cfg.n_q_heads, cfg.head_size, pos)
    x, xb, q, att, out, gate, up = (s[k] for k in ("x", "xb", "q", "att", "out", "gate", "up"))
    x.copy_from(s["embd"].column(int(s["tokens"][0])))
    for l in s["layers"]:
        key, value = l["keys"].column(pos), l["values"].column(pos)
        norm.dispatch(rms, xb, x, l["attn_norm"])
        gemv.dispatch(q, l["attn_q"], xb)
        gemv.dispatch(key, l["attn_k"], xb)
        gemv.dispatch(value, l["attn_v"], xb)
        if case["qwen2"]:
            add.dispatch(q, l["attn_q_bias"])
            add.dispatch(key, l["attn_k_bias"])
            add.dispatch(value, l["attn_v_bias"])
        rope.dispatch(variant, rope_cfg, q, key)
        attention.dispatch_multi(params, q, l["keys"], l["values"], att)
        gemv.dispatch(out, l["attn_output"], att)
        add.dispatch(x, out)
        norm.dispatch(rms, xb, x, l["ffn_norm"])
        gemv.dispatch(gate, l["ffn_gate"], xb)
        gemv.dispatch(up, l["ffn_up"], xb)
        silu.dispatch(gate, up)
        gemv.dispatch(out, l["ffn_down"], gate)
        add.dispatch(x, out)
    norm.dispatch(rms, xb, x, s["output_norm"])
    gemv.dispatch(s["logits"], s["output"], xb)
    return {"token": sampler.sample_argmax(s["logits"]), "logits": s["logits"].read()}


def run(state):
    case = state["case"]
    kind, pos, tokens = case["kind"], case["pos"], state["tokens"]
    if kind == "ops":
        return _run_ops(state)
    m = state["model"]
    if kind == "decode":
        out = m.decode_greedy(int(tokens[0]), pos, case["steps"])
    elif kind == "prompt":
        m.prefill(tokens, pos)
        return {"logits": m.logits()}
    elif kind == "turn":
        m.prefill(tokens, pos)
        first = m.logits()
        out = m.decode_greedy(int(first.argmax()), pos + case["tokens"], case["steps"])
        return {"first": first, "tokens": out, "logits": m.logits()}
    elif kind == "sampled":
        out = m.generate_sampled(tokens, case["tokens"] + case["steps"], 0.8, 0.9, state["seed"] + 5)
    else:
        out = m.generate_greedy(tokens, case["tokens"] + case["steps"])
    return {"tokens": out, "logits": m.logits()}


# ---- what a pass needs ---------------------------------------------------------------------------

def work(case):
    """Bytes: the weights once per decoded token (once for a whole prompt), as stored in the model
    file; the cached rows that attention reads and the new ones; the logits where they are used.
    Flops: two per weight and token, four per query element and attended position."""
    gpt2 = case["kind"] == "gpt2"
    shapes = _gpt2_shapes(case) if gpt2 else _llama_shapes(case)
    layer_elems = sum(r * k for r, k in shapes.values())
    layer_bytes = sum(_file_bytes(_format(case, n, l), r * k)
                      for l in range(case["layers"]) for n, (r, k) in shapes.items())
    out_elems = case["vocab"] * case["dim"]
    out_bytes = _file_bytes(_format(case, "output"), out_elems) + 4 * case["vocab"]
    kv_dim = case["dim"] if gpt2 else case["dim"] // case["heads"] * case["kv_heads"]
    row = 8 * case["layers"] * kv_dim  # K and V of one position, all layers
    total = {"bytes": 0.0, "flops": 0.0}

    def batch(start, n, logits):  # n tokens from position `start` in one pass
        positions = n * start + n * (n + 1) / 2
        total["bytes"] += layer_bytes + row * (start + n) + (out_bytes if logits else 0)
        total["flops"] += 2.0 * n * case["layers"] * layer_elems + (2.0 * out_elems if logits else 0)
        total["flops"] += 4.0 * case["layers"] * case["dim"] * positions

    kind, pos, tokens, steps = case["kind"], case["pos"], case["tokens"], case["steps"]
    if kind in ("prompt", "turn"):
        batch(pos, tokens, True)
        for i in range(steps):
            batch(pos + tokens + i, 1, True)
    elif kind in ("sampled", "gpt2"):
        batch(0, tokens, True)
        for i in range(steps):
            batch(tokens + i, 1, True)
    else:
        for i in range(max(1, steps)):
            batch(pos + i, 1, True)
    return total


def tolerance(case):
    """About four times what other orders of the same sums (attention split differently, K split
    differently, one launch per operator) move the logits by."""
    if case["plain_f16"]:  # operands rounded to 11 bits
        return {"rel": 1e-3, "max": 4e-3, "differ": 0.02}
    if case["scheme"] == "f16" or case["f32_activations"]:
        return {"rel": 3e-6, "max": 1.2e-5, "differ": 0.02}
    if case["kind"] == "prompt":  # fp32-grade products, then one with 16-bit block fixed-point input
        return {"rel": 4e-5, "max": 1.6e-4, "differ": 0.02}
    # every product takes its input as 16-bit block fixed point
    return {"rel": 1.5e-4, "max": 6e-4, "differ": 0.02}

# ---- the same results in 64 bits -----------------------------------------------------------------

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _f64(a):
    return torch.tensor(np.asarray(a), device=_device()).double()


def _half(b, at):
    return b[:, at:at + 2].contiguous().view(torch.float16).double()


def _scales_k(b):  # the 6-bit scales and minima of Q4_K and Q5_K
    lo, mid, hi = b[:, 4:8], b[:, 8:12], b[:, 12:16]
    sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1)
    mn = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1)
    return (_half(b, 0) * sc)[:, :, None], (_half(b, 2) * mn)[:, :, None]


def _dequantize(m):
    """The matrix that the blocks of a GGUF tensor stand for."""
    b = torch.tensor(m.data, device=_device()).reshape(-1, _file_bytes(m.qtype, 256) if m.qtype not in (
        _lib.Q8_0, _lib.Q4_0) else _file_bytes(m.qtype, 32))
    n = len(b)
    if m.qtype == _lib.F16:
        v = b.view(torch.float16).double()
    elif m.qtype == _lib.Q8_0:
        v = _half(b, 0) * b[:, 2:].contiguous().view(torch.int8)
    elif m.qtype == _lib.Q4_0:
        v = _half(b, 0) * (torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8)
    elif m.qtype in (_lib.Q4_K, _lib.Q5_K):
        qs = b[:, -128:].reshape(n, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(n, 8, 32)
        if m.qtype == _lib.Q5_K:
            bit = torch.arange(8, dtype=torch.uint8, device=b.device).reshape(1, 8, 1)
            q = q | (((b[:, None, 16:48] >> bit) & 1) << 4)
        scale, low = _scales_k(b)
        v = scale * q - low
    else:
        ql, qh = b[:, :128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 1, 32)
        shift = torch.arange(0, 8, 2, dtype=torch.uint8, device=b.device).reshape(1, 1, 4, 1)
        q = torch.cat([ql & 15, ql >> 4], 2) | (((qh >> shift) & 3) << 4)
        scale = _half(b, 208) * b[:, 192:208].contiguous().view(torch.int8)
        v = (q.double() - 32).reshape(n, 16, 16) * scale[:, :, None]
    return v.reshape(m.nrows, m.ncols)


class _Exact:
    """A decoder in plain torch and 64 bits: `forward` takes tokens at the next positions and gives
    the last one's logits."""

    def __init__(self, case, host, caches):
        val = lambda v: _dequantize(v) if isinstance(v, HostMatrix) else _f64(v)  # noqa: E731
        self.case, self.gpt2 = case, case["kind"] == "gpt2"
        self.layers = [{k: val(v) for k, v in layer.items()} for layer in host.layers]
        self.caches = caches
        if self.gpt2:
            self.embd, self.pos_embd, self.head = _f64(host.wte), _f64(host.wpe), _dequantize(host.lm_head)
            self.last = (_f64(host.ln_f_g), _f64(host.ln_f_b))
        else:
            self.embd, self.head, self.last = _f64(host.token_embd), _dequantize(host.output), (_f64(host.output_norm),)

    def _norm(self, x, gain, bias=None):
        if bias is None:
            return x / torch.sqrt((x * x).mean(1, keepdim=True) + 1.0e-5) * gain
        x = x - x.mean(1, keepdim=True)
        return x / torch.sqrt((x * x).mean(1, keepdim=True) + 1.0e-5) * gain + bias

    def _rope(self, x, start):
        size = self.case["dim"] // self.case["heads"]
        angle = self.case["rope_base"] ** (-torch.arange(0, size, 2, device=x.device).double() / size)
        angle = (start + torch.arange(len(x), device=x.device).double())[:, None, None] * angle
        c, s = angle.cos(), angle.sin()
        x = x.reshape(len(x), -1, size)
        if self.case["qwen2"]:
            a, b = x[..., :size // 2], x[..., size // 2:]
            return torch.cat([c * a - s * b, s * a + c * b], 2).reshape(len(x), -1)
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([c * a - s * b, s * a + c * b], 3).reshape(len(x), -1)

    def _attention(self, l, q, k, v):
        n, heads = len(q), self.case["heads"]
        size, groups = self.case["dim"] // heads, k.shape[1] // (self.case["dim"] // heads)
        k, v = self.caches[l] = [torch.cat([old, new]) for old, new in zip(self.caches[l], (k, v))]
        q = q.reshape(n, groups, heads // groups, size).permute(1, 2, 0, 3).reshape(groups, -1, size)
        score = torch.matmul(q, k.reshape(-1, groups, size).permute(1, 2, 0).contiguous()) / math.sqrt(size)
        seen = torch.arange(len(k), device=q.device) <= len(k) - n + torch.arange(n, device=q.device)[:, None]
        score = score.reshape(groups, -1, n, len(k)).masked_fill(~seen, -math.inf).softmax(3)
        out = torch.matmul(score.reshape(groups, -1, len(k)), v.reshape(-1, groups, size).permute(1, 0, 2).contiguous())
        return out.reshape(heads, n, size).permute(1, 0, 2).reshape(n, -1)

    def forward(self, tokens, pos):
        x = self.embd[torch.tensor([int(t) for t in tokens], device=self.embd.device)]
        if self.gpt2:
            x = x + self.pos_embd[pos:pos + len(x)]
        for l, w in enumerate(self.layers):
            if self.gpt2:
                qkv = self._norm(x, w["ln_1_g"], w["ln_1_b"]) @ w["attn_w"].T + w["attn_b"]
                x = x + self._attention(l, *qkv.chunk(3, 1)) @ w["attn_proj_w"].T + w["attn_proj_b"]
                h = self._norm(x, w["ln_2_g"], w["ln_2_b"]) @ w["mlp_fc_w"].T + w["mlp_fc_b"]
                h = 0.5 * h * (1 + torch.tanh(math.sqrt(2 / math.pi) * (h + 0.044715 * h ** 3)))
                x = x + h @ w["mlp_proj_w"].T + w["mlp_proj_b"]
                continue
            y = self._norm(x, w["attn_norm"])
            q, k, v = (y @ w["attn_" + n].T + w.get("attn_%s_bias" % n, 0.0) for n in "qkv")
            y = self._attention(l, self._rope(q, pos), self._rope(k, pos), v)
            x = x + y @ w["attn_output"].T
            y = self._norm(x, w["ffn_norm"])
            x = x + (torch.nn.functional.silu(y @ w["ffn_gate"].T) * (y @ w["ffn_up"].T)) @ w["ffn_down"].T
        return (self._norm(x[-1:], *self.last) @ self.head.T)[0].cpu().numpy()


def _sample64(logits, temperature, topp, coin):
    p = np.exp((logits - logits.max()) / temperature)
    p /= p.sum()
    order = np.argsort(-p, kind="stable")
    total = np.cumsum(p[order])
    last = int(np.searchsorted(total, topp, side="right"))  # the first that exceeds topp
    return order[min(last, int(np.searchsorted(total, coin * total[last], side="right")))]


def exact(case, seed):
    """What `run` returns, from the same blocks and vectors."""
    kind, pos, steps = case["kind"], case["pos"], case["steps"]
    tokens = W.rng_tokens(seed + 17, max(1, case["tokens"]), min(SUCCESSORS, case["vocab"]) - 1)
    if kind == "gpt2":
        host, kv, caches = _gpt2_weights(case, seed, _gpt2_params(case)), case["dim"], None
    else:
        cfg = _llama_config(case)
        host, w = _llama_weights(case, seed, cfg)
        kv, caches = cfg.kv_dim, None
        if pos:  # an operator program's caches are filled to their ends
            n = (cfg.seq_len if kind == "ops" else pos) * kv
            caches = [[_f64(w.normal(n)[:pos * kv].reshape(pos, kv)) for _ in range(2)] for _ in host.layers]
    model = _Exact(case, host, caches or [[_f64(np.empty((0, kv)))] * 2 for _ in host.layers])
    if kind == "ops":
        logits = model.forward(tokens, pos)
        return {"token": int(logits.argmax()), "logits": logits}
    if kind == "prompt":
        return {"logits": model.forward(tokens, pos)}
    out, result = [], {}
    if kind == "turn":
        result["first"] = logits = model.forward(tokens, pos)
        pos, token = pos + len(tokens), int(logits.argmax())
    elif kind == "decode":
        token = int(tokens[0])
    else:  # the loops that step through their prompt
        steps, token = len(tokens) + steps, int(tokens[0])
        coins = W.rng_uniform(seed + 5, steps)
    for i in range(steps):
        logits = model.forward([token], pos + i)
        best = int(logits.argmax()) if kind != "sampled" else int(_sample64(logits, 0.8, 0.9, coins[i]))
        token = int(tokens[i + 1]) if kind in ("sampled", "gpt2") and i + 1 < len(tokens) else best
        out.append(best)
    result.update(tokens=np.array(out, np.uint32), logits=logits)
    return result
