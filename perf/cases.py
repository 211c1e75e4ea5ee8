"""Serving work to time: batches of requests with given token ids, through the engine's own steps.

A case is one serving round.  ``batch`` requests of up to ``prompt`` tokens enter in one step (the prompt
pass, the logits of every last prompt token), then ``gen`` steps bring one token per request (decode, the
logits of every row), then the requests end.  ``gen`` 0 is the prompt pass alone.  ``ragged``: the prompts
have different lengths, between half of ``prompt`` and all of it.  The token ids are given, as in a recorded
trace, so a round's logits do not hang on which of two close logits was the larger one.

The models are this repository's presets (full width; ``@<N>l``: that many layers) and the layer-list models
of its throughput benchmark; weights and prompts are random, made on the GPU from the seed.
"""
import json
import math
import os
import tempfile
import zlib

import torch

from distributed_llms_amd.config import EngineConfig, get_model_config
from distributed_llms_amd.engine.hybrid_bench import basopel_config, hybrid_config
from distributed_llms_amd.engine.llm_engine import LLMEngine
from distributed_llms_amd.engine.replay import TraceReplayer
from distributed_llms_amd.models import make_stage
from distributed_llms_amd.models import basopel as basopel_model
from distributed_llms_amd.models import hybrid as tudilix_model

DEVICE = "cuda"


def listed():
    return [
        # one user, a short question, a short answer: the latency of single-token steps
        {"name": "chat_1", "model": "llama3-8b", "batch": 1, "prompt": 37, "ragged": False, "gen": 32, "quant": "none"},
        # a handful of users in different places of their conversations
        {"name": "chat_8", "model": "llama3-8b", "batch": 8, "prompt": 203, "ragged": True, "gen": 16, "quant": "none"},
        # the throughput batch of the headline benchmark: a full decode batch
        {"name": "serve_256", "model": "llama3-8b", "batch": 256, "prompt": 32, "ragged": False, "gen": 24, "quant": "none"},
        # time to the first token of one request
        {"name": "first_token", "model": "llama3-8b", "batch": 1, "prompt": 128, "ragged": False, "gen": 0, "quant": "none"},
        # a step that admits a few waiting requests
        {"name": "admit_24", "model": "llama3-8b", "batch": 24, "prompt": 341, "ragged": True, "gen": 0, "quant": "none"},
        # one long document
        {"name": "document", "model": "llama3-8b", "batch": 1, "prompt": 7937, "ragged": False, "gen": 0, "quant": "none"},
        # the opt-in 8-bit serving mode at a medium batch
        {"name": "fp8_64", "model": "llama3-8b@8l", "batch": 64, "prompt": 40, "ragged": False, "gen": 16, "quant": "fp8"},
        # mixture of experts: a decode batch that touches every expert with few rows each
        {"name": "moe_16", "model": "mixtral-8x7b@4l", "batch": 16, "prompt": 33, "ragged": True, "gen": 24, "quant": "none"},
        # mixture of experts: prompts
        {"name": "moe_prompts", "model": "mixtral-8x7b@4l", "batch": 4, "prompt": 509, "ragged": False, "gen": 0, "quant": "none"},
        # a small recurrent hybrid for one user: every kernel is a few microseconds
        {"name": "hybrid_small_1", "model": "tudilix-small", "batch": 1, "prompt": 21, "ragged": False, "gen": 32, "quant": "none"},
        # the same family at its benchmark size, prompts and answers
        {"name": "hybrid_16", "model": "tudilix-2b", "batch": 16, "prompt": 511, "ragged": True, "gen": 24, "quant": "none"},
        # windows, chunks and latents between layer norms: a medium batch
        {"name": "windows_32", "model": "basopel-2b", "batch": 32, "prompt": 300, "ragged": True, "gen": 24, "quant": "none"},
    ]


# model, largest batch of a drawn decode round, most prompt tokens of a drawn round
DRAWN = [("llama3-8b", 256, 8192), ("llama3-8b", 256, 8192), ("llama3-70b@4l", 256, 4096), ("mixtral-8x7b@4l", 64, 4096),
         ("tudilix-small", 64, 8192), ("tudilix-2b", 64, 16384), ("basopel-small", 64, 8192), ("basopel-2b", 64, 16384)]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    most = max(_seconds(c) for c in listed())
    while True:
        model, batch, tokens = rng.choice(DRAWN)
        c = {"model": model, "batch": _log_uniform(rng, 1, batch), "ragged": rng.random() < 0.5, "quant": "none"}
        if rng.random() < 0.6:                                   # a decode round behind short prompts
            c["gen"] = rng.randint(8, 32)
            c["prompt"] = _log_uniform(rng, 5, max(6, min(512, tokens // c["batch"])))
        else:                                                    # prompts only
            c["gen"] = 0
            c["batch"] = min(c["batch"], 32)
            c["prompt"] = _log_uniform(rng, 9, min(7900, tokens // c["batch"]))
        if model == "llama3-8b" and rng.random() < 0.15:
            c.update(model="llama3-8b@8l", quant="fp8")
        if _seconds(c) <= most:
            return c


# ------------------------------------------------------------------------------ sizes and tokens
def _config(case):
    name = case["model"]
    if name.startswith("tudilix-"):
        return hybrid_config(name.split("-")[1])
    if name.startswith("basopel-"):
        return basopel_config(name.split("-")[1])
    return get_model_config(name)


def _lengths(case):
    b, p = case["batch"], case["prompt"]
    return [p - (i * 7919) % (p // 2 + 1) for i in range(b)] if case["ragged"] else [p] * b


def _tokens(case, seed, vocab):
    g = torch.Generator().manual_seed(int(seed) * 2 + 1)
    return torch.randint(10, vocab - 1, (case["batch"], case["prompt"] + case["gen"]), generator=g)


def _rand(seed, name, shape, scale, shift=0.0):
    g = torch.Generator(DEVICE).manual_seed((int(seed) * 1000003 + zlib.crc32(name.encode())) & 0x7FFFFFFF)
    t = torch.randn(shape, generator=g, device=DEVICE, dtype=torch.bfloat16).mul_(scale)
    return t.add_(shift) if shift else t


def _shapes(cfg):
    """Checkpoint name -> shape."""
    if cfg.arch == "tudilix":
        return tudilix_model.model_shapes(cfg)
    if cfg.arch == "basopel":
        return basopel_model.model_shapes(cfg)
    h, i, v = cfg.hidden_size, cfg.intermediate_size, cfg.vocab_size
    s = {"model.embed_tokens.weight": (v, h), "model.norm.weight": (h,), "lm_head.weight": (v, h)}
    for l in range(cfg.num_layers):
        p = f"model.layers.{l}."
        s.update({p + "input_layernorm.weight": (h,), p + "post_attention_layernorm.weight": (h,),
                  p + "self_attn.q_proj.weight": (cfg.num_heads * cfg.head_dim, h),
                  p + "self_attn.k_proj.weight": (cfg.num_kv_heads * cfg.head_dim, h),
                  p + "self_attn.v_proj.weight": (cfg.num_kv_heads * cfg.head_dim, h),
                  p + "self_attn.o_proj.weight": (h, cfg.num_heads * cfg.head_dim)})
        if cfg.num_experts:
            s[p + "mlp.gate.weight"] = (cfg.num_experts, h)
            s[p + "mlp.experts.gate_up_proj"] = (cfg.num_experts, 2 * i, h)
            s[p + "mlp.experts.down_proj"] = (cfg.num_experts, h, i)
        else:
            s.update({p + "mlp.gate_proj.weight": (i, h), p + "mlp.up_proj.weight": (i, h), p + "mlp.down_proj.weight": (h, i)})
    return s


def _weight(seed, cfg, name, shape):
    """One checkpoint tensor in bfloat16: projections ~ N(0, 1 / fan_in), norms around one, small biases, a router
    wide enough that most choices are not close calls.  Without norms behind the sublayers, the projections into the
    residual stream are scaled down with the depth, as is usual: a layer then adds little to the stream, as it does in
    trained models."""
    leaf = name.rsplit(".", 1)[-1]
    if cfg.arch == "tudilix":
        if leaf == "lam":
            return _rand(seed, name, shape, 1.0, -1.0)
        if leaf == "norm":
            return _rand(seed, name, shape, *((0.1, 0.0) if name == "final.norm" else (0.2, 1.0)))
        if len(shape) == 1 or leaf == "b":
            return _rand(seed, name, shape, 0.1)
        return _rand(seed, name, shape, 1.0 if name == "embed" else shape[-1] ** -0.5)
    if cfg.arch == "basopel":
        if leaf in ("norm", "norm1", "norm1b", "norm2", "norm2b"):
            return _rand(seed, name, shape, 0.2, 1.0)
        if leaf == "b":
            return _rand(seed, name, shape, 0.1)
        if leaf == "vmix":
            return _rand(seed, name, shape, 0.1, 0.5)
        return _rand(seed, name, shape, 1.0 if leaf in ("rel", "sink") else shape[-1] ** -0.5)
    if len(shape) == 1:
        return _rand(seed, name, shape, 0.2, 1.0)
    if name.endswith("mlp.gate.weight"):
        return _rand(seed, name, shape, 3.0 * shape[-1] ** -0.5)
    if "o_proj" in name or "down_proj" in name and "gate_up" not in name:
        return _rand(seed, name, shape, 0.125 * shape[-1] ** -0.5)
    return _rand(seed, name, shape, 1.0 if "embed" in name else shape[-1] ** -0.5)


# ------------------------------------------------------------------------------ a round
def prepare(case, seed):
    cfg = _config(case)
    b, p, gen = case["batch"], case["prompt"], case["gen"]
    stage = make_stage(cfg, device=DEVICE, dtype=torch.bfloat16)
    stage.load_hf_state({n: _weight(seed, cfg, n, s) for n, s in _shapes(cfg).items()})
    stage.quantize(case["quant"])
    lens = _lengths(case)
    kw = {}
    if cfg.is_layer_list:
        kw["shard_dir"] = tempfile.mkdtemp(prefix="dllm_cases_")
        with open(os.path.join(kw["shard_dir"], "config.json"), "w") as f:
            json.dump(cfg.to_hf_config(), f)
    ecfg = EngineConfig(model=case["model"], device=DEVICE, dtype="bfloat16", max_batch=b, max_seq_len=p + gen + 8,
                        num_kv_blocks=sum(-(-(n + gen) // 32) for n in lens) + b + 2, max_prefill_tokens=max(16384, b * p),
                        quant=case["quant"], **kw)
    eng = LLMEngine(ecfg, stage)
    if gen:                                          # the graphs of the decode steps, as a server's warm-up makes them
        eng.runner.warmup_graphs([b], sorted({eng.runner.graphs.bucket(b, max(lens) + k)[1] for k in range(1, gen + 1)}))
    toks = _tokens(case, seed, cfg.vocab_size).tolist()
    torch.cuda.synchronize()
    return {"replayer": TraceReplayer(eng), "prompts": [t[:n] for t, n in zip(toks, lens)],
            "answers": [t[n:n + gen] for t, n in zip(toks, lens)], "gen": gen}


def run(state):
    rp, gen = state["replayer"], state["gen"]
    names = [f"request{i}" for i in range(len(state["prompts"]))]
    out = [rp.step([(n, t, [len(t) - 1]) for n, t in zip(names, state["prompts"])], end=() if gen else names)]
    for k in range(gen):
        out.append(rp.step([(n, [t[k]], [0]) for n, t in zip(names, state["answers"])], end=names if k == gen - 1 else ()))
    return out


def work(case):
    """Every step reads the weights it needs once (all of them; of the experts as many as can be chosen), a decode step
    the visible keys and values of every row, and every new key, value and wanted logit is written once."""
    cfg = _config(case)
    lens, gen = _lengths(case), case["gen"]
    b, n = len(lens), sum(lens)
    v, h = cfg.vocab_size, cfg.hidden_size
    heads, kv, spans = _attention_sizes(cfg)
    dense, expert = _layer_params(cfg)
    el = 1 if case["quant"] == "fp8" else 2

    def step_bytes(rows):
        touched = expert * min(cfg.num_experts, rows * cfg.experts_per_token) if expert else 0
        return (dense + touched) * el + v * h * 2 + b * v * 4 + rows * h * 2 + rows * kv * 2

    pairs = 0                                        # multiply-adds of the scores and of their sums
    nbytes = step_bytes(n) + sum(step_bytes(b) for _ in range(gen))
    for width, span, kvw in spans:
        for t in lens:
            seen = min(t, span)
            pairs += width * (seen * (seen + 1) // 2 + (t - seen) * seen)
            for k in range(1, gen + 1):
                pairs += width * min(t + k, span)
                nbytes += kvw * 2 * min(t + k, span)
    active = dense + expert * cfg.experts_per_token
    flops = 2 * active * (n + b * gen) + 2 * v * h * b * (gen + 1) + 2 * pairs
    return {"bytes": float(nbytes), "flops": float(flops)}


def _attention_sizes(cfg):
    """(query heads, cached values per token over all layers, per attention layer (multiply-adds per seen key, largest
    number of seen keys, cached values per key))."""
    if not cfg.is_layer_list:
        kvw = 2 * cfg.num_kv_heads * cfg.head_dim
        return cfg.num_heads, kvw * cfg.num_layers, [(cfg.num_heads * 2 * cfg.head_dim, 1 << 30, kvw)] * cfg.num_layers
    spans = []
    for l in cfg.layers:
        m = l["mixer"]
        if l["type"] == "rglru":
            continue
        size = (m.get("mask") or {}).get("size", 1 << 30)
        if l["type"] == "latent_attention":
            spans.append((m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"]), size, m["kv_rank"] + m["rot_dim"]))
        else:
            spans.append((m["heads"] * (m["dim"] + m["vdim"]), size, m["kv_heads"] * (m["dim"] + m["vdim"])))
    return cfg.num_heads, sum(s[2] for s in spans), spans


def _layer_params(cfg):
    """(weights every token uses, weights of one expert) over all layers, without embedding and head."""
    dense = expert = 0
    for name, shape in _shapes(cfg).items():
        if name.startswith(("model.embed", "model.norm", "lm_head", "embed", "final", "head")):
            continue
        n = math.prod(shape)
        if ".experts." in name:
            expert += n // shape[0]
        else:
            dense += n
    return dense, expert


def _seconds(case):
    w = work(case)
    return w["bytes"] / 4e12 + w["flops"] / 1e15 + 2e-4 * (1 + case["gen"])


def tolerance(case):
    """bfloat16 activations between the layers.  Two orders of the sums (other splits of the reductions, other kernels)
    give logits that are 0.006 to 0.013 of their size apart, 0.07 at most in one value; where an expert's choice or an
    8-bit rounding falls the other way, 0.02 and 0.24."""
    return {"rel": 0.03, "max": 0.5}


# ------------------------------------------------------------------------------ the same in 64 bits
def exact(case, seed):
    """The logits of whole sequences, computed at once: what the steps return, position by position."""
    if _seconds(case) > 2.0:
        return None
    cfg = _config(case)
    lens, gen = _lengths(case), case["gen"]
    toks = _tokens(case, seed, cfg.vocab_size).to(DEVICE)
    shapes = _shapes(cfg)

    def w(name):
        return _weight(seed, cfg, name, shapes[name]).double()

    with torch.inference_mode():
        forward = {"tudilix": _tudilix, "basopel": _basopel}.get(cfg.arch, _llama)
        x, head = forward(cfg, w, toks, case["quant"] == "fp8")
        rows = torch.arange(len(lens), device=DEVICE)
        at = torch.tensor(lens, device=DEVICE) - 1
        return [head(x[rows, at + k]) for k in range(gen + 1)]


def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _layer_norm(x, w, b, eps):
    c = x - x.mean(-1, keepdim=True)
    return _rms(c, eps) * w + b


def _gelu(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def _rotate(x, inv, mag=1.0, halves=True):
    """x [B, T, H, D]: the first 2 len(inv) dimensions turn, as two halves or as neighbouring pairs."""
    a = torch.arange(x.shape[1], device=x.device, dtype=torch.float64)[:, None] * inv.to(x.device)[None]
    c, s, n = (a.cos() * mag)[:, None], (a.sin() * mag)[:, None], inv.numel()
    out = x.clone()
    if halves:
        u, v = x[..., :n], x[..., n:2 * n]
        out[..., :n], out[..., n:2 * n] = u * c - v * s, v * c + u * s
    else:
        u, v = x[..., 0:2 * n:2], x[..., 1:2 * n:2]
        out[..., 0:2 * n:2], out[..., 1:2 * n:2] = u * c - v * s, v * c + u * s
    return out


def _attend(q, k, v, scale, sees=None, cap=0.0, bias=None, sink=None):
    """Causal softmax attention, q [B, T, H, D], k / v [B, T, G, .]; ``sees(i, j)``: which of the earlier positions j a
    query at i sees; ``bias`` [T, H] by distance; ``sink`` [H] joins the denominator."""
    b, t, h, _ = q.shape
    rep = h // k.shape[2]
    out = torch.empty(b, t, h, v.shape[-1], dtype=q.dtype, device=q.device)
    nh = max(1, min(h, (1 << 28) // (t * t))) if t * t * h > 1 << 28 else h
    nb = max(1, (1 << 28) // (t * t * nh))
    j = torch.arange(t, device=q.device)
    ok = j[None, :] <= j[:, None]
    if sees is not None:
        ok = ok & sees(j[:, None], j[None, :])
    for b0 in range(0, b, nb):
        for h0 in range(0, h, nh):
            hs = torch.arange(h0, min(h, h0 + nh), device=q.device)
            qq = q[b0:b0 + nb, :, hs].transpose(1, 2).contiguous()
            kk = k[b0:b0 + nb, :, hs // rep].permute(0, 2, 3, 1).contiguous()
            vv = v[b0:b0 + nb, :, hs // rep].transpose(1, 2).contiguous()
            s = torch.matmul(qq, kk).mul_(scale)
            if cap:
                s = cap * torch.tanh(s / cap)
            if bias is not None:
                s += bias[(j[:, None] - j[None, :]).clamp_(min=0)][:, :, hs].permute(2, 0, 1)
            s.masked_fill_(~ok, -math.inf)
            top = s.amax(-1, keepdim=True)
            if sink is not None:
                top = torch.maximum(top, sink[hs][None, :, None, None])
            s = s.sub_(top).exp_()
            den = s.sum(-1, keepdim=True)
            if sink is not None:
                den = den + (sink[hs][None, :, None, None] - top).exp()
            out[b0:b0 + nb, :, hs] = (torch.matmul(s, vv) / den).transpose(1, 2)
    return out


def _llama3_frequencies(cfg):
    d = cfg.head_dim
    inv = cfg.rope_theta ** (-torch.arange(0, d, 2, dtype=torch.float64) / d)
    r = cfg.rope_scaling
    if r:
        length = 2 * math.pi / inv
        lo, hi = r["original_max_position_embeddings"] / r["low_freq_factor"], r["original_max_position_embeddings"] / r["high_freq_factor"]
        f = (r["original_max_position_embeddings"] / length - r["low_freq_factor"]) / (r["high_freq_factor"] - r["low_freq_factor"])
        mid = (1 - f) * inv / r["factor"] + f * inv
        inv = torch.where(length > lo, inv / r["factor"], torch.where(length < hi, inv, mid))
    return inv


def _e4m3(w):
    """Rows rounded to 8 bits under one scale each."""
    s = (w.abs().amax(1, keepdim=True).float() / 448.0).clamp_min(1e-12)
    return ((w.float() / s).to(torch.float8_e4m3fn).float() * s).double()


def _llama(cfg, w, toks, fp8):
    eps, (b, t) = cfg.norm_eps, toks.shape
    inv = _llama3_frequencies(cfg)
    x = w("model.embed_tokens.weight")[toks]
    m = (lambda n: _e4m3(w(n))) if fp8 else w
    for l in range(cfg.num_layers):
        p = f"model.layers.{l}."
        h = _rms(x, eps) * w(p + "input_layernorm.weight")
        q, k, v = ((h @ m(p + f"self_attn.{c}_proj.weight").T).view(b, t, -1, cfg.head_dim) for c in "qkv")
        o = _attend(_rotate(q, inv), _rotate(k, inv), v, cfg.head_dim ** -0.5)
        x = x + o.view(b, t, -1) @ m(p + "self_attn.o_proj.weight").T
        h = _rms(x, eps) * w(p + "post_attention_layernorm.weight")
        silu = torch.nn.functional.silu
        if not cfg.num_experts:
            x = x + (silu(h @ m(p + "mlp.gate_proj.weight").T) * (h @ m(p + "mlp.up_proj.weight").T)) @ m(p + "mlp.down_proj.weight").T
            continue
        h = h.view(b * t, -1)
        top, idx = (h @ w(p + "mlp.gate.weight").T).softmax(-1).topk(cfg.experts_per_token, -1)
        top = top / top.sum(-1, keepdim=True)
        gu, dn = w(p + "mlp.experts.gate_up_proj"), w(p + "mlp.experts.down_proj")
        y = torch.zeros_like(h)
        for e in range(cfg.num_experts):
            r, c = (idx == e).nonzero(as_tuple=True)
            g, u = (h[r] @ gu[e].T).chunk(2, -1)
            y.index_add_(0, r, (silu(g) * u) @ dn[e].T * top[r, c][:, None])
        x = x + y.view(b, t, -1)
    fn, head = w("model.norm.weight"), w("lm_head.weight")
    return x, lambda r: (_rms(r, eps) * fn) @ head.T


def _tudilix(cfg, w, toks, _fp8):
    eps, (b, t) = cfg.norm_eps, toks.shape

    def conv(u, c):                                  # c [C, taps]; zeros before the first position
        n = c.shape[1]
        return sum(torch.nn.functional.pad(u, (0, 0, n - 1 - j, 0))[:, :t] * c[:, j] for j in range(n))

    def frequencies(r):
        d, base = r["dims"], r["base"]
        f, mag, sc = [base ** (-2.0 * i / d) for i in range(d // 2)], 1.0, r.get("scaling")
        if sc:
            at = [d * math.log(sc["original"] / (2 * math.pi * n)) / (2 * math.log(base)) for n in (sc["fast"], sc["slow"])]
            lo, hi = max(math.floor(at[0]), 0), min(math.ceil(at[1]), d - 1)
            ramp = [min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0) for i in range(d // 2)]
            f = [a / sc["factor"] * s + a * (1 - s) for a, s in zip(f, ramp)]
            mag = 0.1 * math.log(sc["factor"]) + 1.0
        return torch.tensor(f, dtype=torch.float64), mag

    norm = lambda z, n: _rms(z, eps) * (1.0 + w(n))
    x = w("embed")[toks]
    for i, layer in enumerate(cfg.layers):
        p, m = f"l{i}.", layer["mixer"]
        h = norm(x, p + "norm1")
        if layer["type"] == "attention":
            q, k, v = (conv(h @ w(p + f"mix.{c}").T, w(p + f"mix.{c}.conv")).view(b, t, -1, m["vdim" if c == "v" else "dim"]) for c in "qkv")
            q, k = (_rotate(_rms(z, eps) * w(p + f"mix.{c}.norm"), *frequencies(m["rot"]), halves=False) for z, c in ((q, "q"), (k, "k")))
            o = _attend(q, k, v, m["scale"], lambda a, c: a - c < m["mask"]["size"]).view(b, t, -1)
        else:
            y = _gelu(h @ w(p + "mix.y").T + w(p + "mix.y.b"))
            u = conv(h @ w(p + "mix.x").T + w(p + "mix.x.b"), w(p + "mix.conv")) + w(p + "mix.conv.b")
            ub = u.view(b * t, m["blocks"], -1).transpose(0, 1).contiguous()
            r, g = (torch.sigmoid(torch.matmul(ub, w(p + f"mix.{c}").transpose(1, 2).contiguous()) + w(p + f"mix.{c}.b")[:, None])
                    .transpose(0, 1).reshape(b, t, -1) for c in ("ra", "ri"))
            a = torch.exp(-8.0 * r * torch.nn.functional.softplus(w(p + "mix.lam")))
            z = torch.sqrt(1.0 - a * a) * g * u
            s = torch.zeros_like(z[:, 0])
            for j in range(t):
                s = a[:, j] * s + z[:, j]
                z[:, j] = s
            o = z * y
        x = x + cfg.residual_mult * norm(o @ w(p + "mix.o").T, p + "norm1b")
        if layer.get("mlp"):
            h, c = norm(x, p + "norm2"), layer["mlp"]["limit"]
            g = (h @ w(p + "mlp.gate").T + w(p + "mlp.gate.b")).clamp(max=c)
            u = (h @ w(p + "mlp.up").T + w(p + "mlp.up.b")).clamp(-c, c)
            y = (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ w(p + "mlp.down").T + w(p + "mlp.down.b")
            x = x + cfg.residual_mult * norm(y, p + "norm2b")
    fn, head, cap = 1.0 + w("final.norm"), w("head"), cfg.logit_softcap

    def logits(r):
        z = (_rms(r, eps) * fn) @ head.T
        return cap * torch.tanh(z / cap) if cap else z
    return x, logits


def _basopel(cfg, w, toks, _fp8):
    eps, (b, t) = cfg.norm_eps, toks.shape
    norm = lambda z, n: _layer_norm(z, w(n), w(n + ".b"), eps)

    def frequencies(r):
        f = r["base"] ** (-2.0 * torch.arange(r["dims"] // 2, dtype=torch.float64) / r["dims"])
        return f / (r.get("scaling") or {}).get("factor", 1.0)

    def biases(rel, far):                            # one row per distance
        rows, half = rel.shape[0], rel.shape[0] // 2
        row = [n if n < half else min(rows - 1, half + math.floor(math.log(n / half) / math.log(far / half) * (rows - half)))
               for n in range(t)]
        return rel[torch.tensor(row, device=rel.device)]

    x = w("embed")[toks] * cfg.embed_scale
    first = None                                     # the values of the first layer that shares them
    for i, layer in enumerate(cfg.layers):
        p, q_, m = f"l{i}.", f"l{i}.mix.", layer["mixer"]
        h, size = norm(x, p + "norm1"), m["mask"]["size"]
        if layer["type"] == "latent_attention":
            hh, r, d = m["heads"], m["kv_rank"], m["dim"]
            q = (h @ w(q_ + "q").T).view(b, t, hh, -1)
            kv = h @ w(q_ + "dkv").T
            c = _rms(kv[..., :r], eps) * w(q_ + "dkv.norm")
            inv = frequencies(m["rot"])
            q = torch.cat([q[..., :d], _rotate(q[..., d:], inv)], -1)
            k = torch.cat([(c @ w(q_ + "uk").T).view(b, t, hh, d), _rotate(kv[:, :, None, r:], inv).expand(b, t, hh, -1)], -1)
            v = (c @ w(q_ + "uv").T).view(b, t, hh, -1)
            o = _attend(q, k, v, m["scale"], lambda a, c: a - c < size, sink=w(q_ + "sink")).view(b, t, -1)
            o = (o * torch.sigmoid(h @ w(q_ + "g").T)) @ w(q_ + "o").T
        else:
            q, k, v = (h @ w(q_ + c).T + w(q_ + c + ".b") for c in "qkv")
            if m.get("v_mix"):
                if first is None:
                    first = v
                else:
                    lam = w(q_ + "vmix")
                    v = (1.0 - lam) * v + lam * first
            v = v.view(b, t, m["kv_heads"], -1)
            if layer["type"] == "attention":
                q, k = (_rms(z.view(b, t, -1, m["dim"]), eps) * w(q_ + c + ".norm") for z, c in ((q, "q"), (k, "k")))
                keep = m["mask"]["keep_first"]
                o = _attend(q, k, v, m["scale"], lambda a, c: (a - c < size) | (c < keep), bias=biases(w(q_ + "rel"), m["bias_max"]))
                o = o.view(b, t, -1) @ w(q_ + "o").T
            else:
                inv = frequencies(m["rot"])
                q, k = (_rotate((_rms(z, eps) * w(q_ + c + ".norm")).view(b, t, -1, m["dim"]), inv) for z, c in ((q, "q"), (k, "k")))
                o = _attend(q, k, v, m["scale"], lambda a, c: a // size == c // size, cap=m["softcap"], sink=w(q_ + "sink"))
                o = o * torch.sigmoid(h @ w(q_ + "g").T)[..., None]
                o = o.view(b, t, -1) @ w(q_ + "o").T + w(q_ + "o.b")
        x = x + norm(o, p + "norm1b")
        if layer.get("mlp"):
            h = norm(x, p + "norm2")
            y = (_gelu(h @ w(p + "mlp.gate").T) * (h @ w(p + "mlp.up").T)) @ w(p + "mlp.down").T
            x = x + norm(y, p + "norm2b")
    fw, fb, head = w("final.norm"), w("final.norm.b"), w("embed")
    return x, lambda r: _layer_norm(r, fw, fb, eps) @ head.T
