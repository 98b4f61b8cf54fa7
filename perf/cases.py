"""What is timed of the serving path, and what its outputs are held against.

A case is one pass of the model runner (or, for the family with recurrent
state, of the engine) over a batch as the scheduler forms it: decode steps
of one to 256 requests, prompts, prompt portions behind a cached context,
and the mixed step in which new prompts join the running requests. Models
are the registry's Qwen3-8B and Qwen3-30B-A3B with their own layer and
vocabulary sizes and the design that ``bench.py --mixer-compare`` names
Vatunex; the number of layers is cut so that weights are drawn quickly.
Weights arrive as checkpoint tensors through the loader, contexts through
the cache op, block ids are scattered as in a server that has run a while.
"""

import itertools
import math
import random
import zlib

import torch

import fusioninfer_amd.ops as ops
from fusioninfer_amd.config import CacheConfig, EngineConfig, SchedulerConfig
from fusioninfer_amd.engine.block_manager import BlockManager
from fusioninfer_amd.engine.llm_engine import LLMEngine
from fusioninfer_amd.engine.model_runner import ModelRunner
from fusioninfer_amd.engine.sequence import SamplingParams, Sequence
from fusioninfer_amd.models.registry import (
    get_model_config,
    model_config_from_dict,
)
from fusioninfer_amd.models.weight_loader import load_hf_state_dict

DEV = "cuda:0"
F64 = torch.float64
F8 = torch.float8_e4m3fn
BLOCK = 16
LAYERS = {"Qwen3-8B": 8, "Qwen3-30B-A3B": 4, "Vatunex": 4}


# ------------------------------------------------------------------ cases

def _case(name, model, decode=0, ctx=(0, 0), prompts=0, new=(0, 0), past=0,
          fp8=False, fp8_kv=False, steps=0):
    """decode: requests that decode one token each, at contexts of ctx[0]
    to ctx[1] tokens; prompts: requests with new[0] to new[1] prompt tokens
    in this step, behind ``past`` tokens already in the cache; steps: tokens
    decoded after the prompts within the pass (Vatunex)."""
    c = {"model": model, "decode": decode, "ctx_lo": ctx[0],
         "ctx_hi": ctx[1], "prompts": prompts, "new_lo": new[0],
         "new_hi": new[1], "past": past, "fp8": fp8, "fp8_kv": fp8_kv,
         "steps": steps}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one chat user: every generated token is such a step
        _case("decode_one", "Qwen3-8B", decode=1, ctx=(301, 301)),
        # a few users at very different points of their conversations
        _case("decode_few", "Qwen3-8B", decode=13, ctx=(70, 4100)),
        # the serving benchmark's full house (1024-token prompts, answers
        # of up to 256 tokens)
        _case("decode_full", "Qwen3-8B", decode=256, ctx=(1024, 1279)),
        # long documents, few users
        _case("decode_long", "Qwen3-8B", decode=6, ctx=(20011, 32700)),
        # the fp8 serving mode with the fp8 cache, moderate load
        _case("decode_fp8", "Qwen3-8B", decode=64, ctx=(512, 2048),
              fp8=True, fp8_kv=True),
        # mixture-of-experts decode, moderate load
        _case("decode_moe", "Qwen3-30B-A3B", decode=64, ctx=(512, 2048)),
        # a short question arrives at an idle server: time to first token
        _case("prompt_short", "Qwen3-8B", prompts=1, new=(43, 43)),
        # the serving benchmark's admission step: new prompts up to the
        # token budget join the running requests
        _case("admission", "Qwen3-8B", decode=243, ctx=(1024, 1279),
              prompts=7, new=(900, 1200)),
        # one portion of a long document behind what is already cached
        _case("portion", "Qwen3-8B", prompts=1, new=(4099, 4099),
              past=16384),
        # prompts in the fp8 serving mode
        _case("prompts_fp8", "Qwen3-8B", prompts=8, new=(512, 1500),
              fp8=True, fp8_kv=True),
        # prompts of the mixture of experts
        _case("prompts_moe", "Qwen3-30B-A3B", prompts=8, new=(512, 1500)),
        # whole requests of the recurrent/latent design: prompts, then
        # tokens one by one
        _case("vatunex_requests", "Vatunex", prompts=4, new=(1500, 2048),
              steps=8),
    ]


def _log_int(rng, lo, hi):
    return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prompts", "prompts",
                       "mixed", "vatunex"])
    if kind == "vatunex":
        hi = _log_int(rng, 30, 2048)
        return _case(None, "Vatunex", prompts=rng.randint(1, 4),
                     new=(max(1, hi * 2 // 3), hi), steps=rng.randint(1, 8))
    model = rng.choice(["Qwen3-8B", "Qwen3-8B", "Qwen3-30B-A3B"])
    fp8 = model == "Qwen3-8B" and rng.random() < 0.35
    fp8_kv = rng.random() < (0.7 if fp8 else 0.15)
    decode, prompts, past, ctx, new = 0, 0, 0, (0, 0), (0, 0)
    if kind in ("decode", "mixed"):
        decode = _log_int(rng, 1, 256)
        hi = _log_int(rng, 40, min(32700, 300000 // decode))
        ctx = (max(17, int(hi * rng.uniform(0.1, 1.0))), hi)
        ctx = (min(ctx), hi)
    if kind in ("prompts", "mixed"):
        prompts = _log_int(rng, 1, 8)
        hi = _log_int(rng, 5, 8192 // prompts)
        new = (max(1, hi * 2 // 3), hi)
        if rng.random() < 0.3:
            past = _log_int(rng, 16, 16384 // prompts)
    return _case(None, model, decode, ctx, prompts, new, past, fp8, fp8_kv)


def _lengths(case):
    """(contexts of the decoding requests, prompt lengths), from the case
    alone."""
    rng = random.Random(7 * case["decode"] + case["ctx_hi"])
    ctx = [rng.randint(case["ctx_lo"], case["ctx_hi"])
           for _ in range(case["decode"])]
    new = [rng.randint(case["new_lo"], case["new_hi"])
           for _ in range(case["prompts"])]
    return ctx, new


# ---------------------------------------------------------------- weights

def _gen(seed, tag):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) << 32) + zlib.crc32(tag.encode()))
    return g


def _normal(seed, tag, shape, std=0.02, mean=0.0):
    t = torch.empty(shape, dtype=torch.bfloat16, device=DEV)
    return t.normal_(mean, std, generator=_gen(seed, tag))


def _uniform(seed, tag, shape, lo, hi):
    t = torch.empty(shape, dtype=torch.float32, device=DEV)
    return t.uniform_(lo, hi, generator=_gen(seed, tag))


# Sublayers add to a stream that is larger than what one of them adds (their
# last matrix is drawn smaller by the root of the number of sublayers), and
# head norms sharpen attention to a handful of keys, as in trained models.
EMBED_STD = 1.5
OUT_STD = 0.02 / math.sqrt(72.0)
HEAD_NORM = 1.25


def _projection(case, seed, name, shape, std=0.02):
    """Checkpoint tensors of one projection: bf16, or e4m3 with a scale per
    output row."""
    w = _normal(seed, name, shape, std)
    if not case["fp8"]:
        return [(name + ".weight", w)]
    scale = w.abs().amax(dim=1).float() / 448.0
    return [(name + ".weight", (w.float() / scale[:, None]).to(F8)),
            (name + ".weight_scale", scale)]


def _layer_tensors(case, mc, seed, i):
    h, p = mc.hidden_size, f"model.layers.{i}."
    for n in ("input_layernorm", "post_attention_layernorm"):
        yield p + n + ".weight", _normal(seed, p + n, (h,), 0.1, 1.0)
    for n in ("q", "k"):
        yield (p + f"self_attn.{n}_norm.weight",
               _normal(seed, p + n + "n", (mc.head_dim,), 0.1, HEAD_NORM))
    for n, rows in (("q", mc.q_size), ("k", mc.kv_size), ("v", mc.kv_size)):
        yield from _projection(case, seed, p + f"self_attn.{n}_proj",
                               (rows, h))
    yield from _projection(case, seed, p + "self_attn.o_proj",
                           (h, mc.q_size), OUT_STD)
    if not mc.is_moe:
        f = mc.intermediate_size
        for n, shape, std in (("gate", (f, h), 0.02), ("up", (f, h), 0.02),
                              ("down", (h, f), OUT_STD)):
            yield from _projection(case, seed, p + f"mlp.{n}_proj", shape,
                                   std)
        return
    f, e = mc.moe_intermediate_size, mc.num_experts
    yield p + "mlp.gate.weight", _normal(seed, p + "router", (e, h))
    gate = _normal(seed, p + "gate", (e, f, h))
    up = _normal(seed, p + "up", (e, f, h))
    down = _normal(seed, p + "down", (e, h, f), OUT_STD)
    for j in range(e):
        q = p + f"mlp.experts.{j}."
        yield q + "gate_proj.weight", gate[j]
        yield q + "up_proj.weight", up[j]
        yield q + "down_proj.weight", down[j]


def _outer_tensors(mc, seed):
    v, h = mc.vocab_size, mc.hidden_size
    yield "model.embed_tokens.weight", _normal(seed, "embed", (v, h),
                                               EMBED_STD)
    yield "lm_head.weight", _normal(seed, "head", (v, h))
    yield "model.norm.weight", _normal(seed, "norm", (h,), 0.1, 1.0)


def _context(mc, seed, layer, which, tokens):
    """Cached rows: keys are normed per head, values are projections of
    normed rows."""
    std = HEAD_NORM if which == "k" else 0.02 * math.sqrt(mc.hidden_size)
    return _normal(seed, f"ctx{layer}{which}", (tokens, mc.kv_size), std)


def _tokens(case, seed, vocab):
    ctx, new = _lengths(case)
    rng = random.Random(seed)
    last = [rng.randrange(vocab) for _ in ctx]
    prompts = [[rng.randrange(vocab) for _ in range(n + case["steps"])]
               for n in new]
    return ctx, new, last, prompts


# ---------------------------------------------------------------- prepare

def _model(case):
    if case["model"] == "Vatunex":
        mc = model_config_from_dict(_vatunex())
        mc.name = "vatunex-2048x16"
        return mc
    mc = get_model_config(case["model"])
    # e4m3 rounding decides otherwise after any other bf16 rounding, layer
    # by layer; two layers keep outputs comparable
    mc.num_layers = min(LAYERS[case["model"]], 2 if case["fp8"] else 99)
    mc.quantization = "fp8" if case["fp8"] else None
    return mc


def _engine_config(case, mc, ctx, new):
    rows = [c + BLOCK for c in ctx] + \
        [case["past"] + n + case["steps"] + BLOCK for n in new]
    longest = max(rows)
    blocks = sum(r // BLOCK + 1 for r in rows) + 8
    return EngineConfig(
        model=mc,
        cache=CacheConfig(
            block_size=BLOCK, num_gpu_blocks=blocks,
            kv_cache_dtype="fp8" if case["fp8_kv"] else "auto",
            enable_prefix_caching=False),
        scheduler=SchedulerConfig(
            max_num_seqs=1 << (max(len(ctx), len(new)) - 1).bit_length(),
            max_model_len=8192 if longest <= 8192 else 40960),
        # a step with prompts is launched op by op; decode graphs would be
        # captured for nothing
        enforce_eager=not (ctx and not new) and not case["steps"],
        seed=1)


def prepare(case, seed):
    mc = _model(case)
    ctx, new, last, prompts = _tokens(case, seed, mc.vocab_size)
    cfg = _engine_config(case, mc, ctx, new)
    if case["model"] == "Vatunex":
        engine = LLMEngine(cfg, DEV)
        engine.runner.model.load_weights(_vatunex_tensors(seed))
        return {"engine": engine, "new": new, "prompts": prompts,
                "steps": case["steps"]}
    runner = ModelRunner(cfg, DEV)
    experts = [m for m in runner.model.modules()
               if hasattr(m, "ensure_unpacked")]
    for m in experts:
        m.ensure_unpacked()
    load_hf_state_dict(runner.model, itertools.chain(
        _outer_tensors(mc, seed),
        *(_layer_tensors(case, mc, seed, i) for i in range(mc.num_layers))))
    for m in experts:
        m.release_unpacked()
    runner.allocate_kv_caches()
    bm = BlockManager(runner.num_gpu_blocks, BLOCK)
    random.Random(seed).shuffle(bm.free_blocks)
    decoding, joining, slots = [], [], []
    for i, (n, t) in enumerate(zip(ctx, last)):
        # n tokens in the cache, the one sampled last is decoded now
        s = Sequence(f"d{i}", [1] * n, SamplingParams())
        bm.allocate(s)
        slots += [bm.slot_for(s, j) for j in range(n)]
        s.num_computed_tokens = n
        s.append_token(t)
        bm.append_slot(s)
        decoding.append(s)
    for i, p in enumerate(prompts):
        s = Sequence(f"p{i}", [1] * case["past"] + p, SamplingParams())
        bm.allocate(s)
        slots += [bm.slot_for(s, j) for j in range(case["past"])]
        s.num_computed_tokens = case["past"]
        joining.append(s)
    if slots:
        at = torch.tensor(slots, dtype=torch.int32, device=DEV)
        for i, (k, v) in enumerate(runner.kv_caches):
            ops.reshape_and_cache(_context(mc, seed, i, "k", len(slots)),
                                  _context(mc, seed, i, "v", len(slots)),
                                  k, v, at)
    runner.capture_decode_graphs()
    return {"runner": runner, "bm": bm, "decode": decoding,
            "prompts": joining, "new": new}


# -------------------------------------------------------------------- run

def run(state):
    """The logits of every sampled row."""
    if "engine" in state:
        return _run_requests(state)
    runner, bm = state["runner"], state["bm"]
    if not state["prompts"]:
        return runner.execute_decode(state["decode"], bm)
    if not state["decode"]:
        return runner.execute_prefill(state["prompts"], bm)
    return runner.run_batch(runner.build_batch_payload(
        state["prompts"], state["new"], state["decode"], bm))


def _run_requests(state):
    engine, new, prompts = state["engine"], state["new"], state["prompts"]
    ids = [f"r{i}" for i in range(len(new))]
    out = [engine.forced_step([(r, p[:n], [n - 1])
                               for r, n, p in zip(ids, new, prompts)])]
    for t in range(state["steps"]):
        out.append(engine.forced_step(
            [(r, [p[n + t]], [0]) for r, n, p in zip(ids, new, prompts)],
            ids if t + 1 == state["steps"] else ()))
    return out


# ------------------------------------------------------------------- work

def work(case):
    ctx, new = _lengths(case)
    if case["model"] == "Vatunex":
        return _vatunex_work(case, new)
    mc = _model(case)
    L, h, f = mc.num_layers, mc.hidden_size, mc.intermediate_size
    T = len(ctx) + sum(new)
    S = len(ctx) + len(new)
    wb = 1 if case["fp8"] else 2
    attn = h * (mc.q_size + 2 * mc.kv_size) + mc.q_size * h
    if mc.is_moe:
        e, k, f = mc.num_experts, mc.num_experts_per_tok, \
            mc.moe_intermediate_size
        touched = e * (1.0 - (1.0 - k / e) ** T)
        active, read = attn + e * h + 3 * h * f * k, \
            attn + e * h + 3 * h * f * touched
    else:
        active = read = attn + 3 * h * f
    # (row, visible key) pairs and cached rows that are read
    pairs = sum(c + 1 for c in ctx) + \
        sum(n * case["past"] + n * (n + 1) // 2 for n in new)
    held = sum(ctx) + case["past"] * len(new)
    kvb = 1 if case["fp8_kv"] else 2
    flops = 2 * L * T * active + 4 * L * mc.q_size * pairs + \
        2 * S * h * mc.vocab_size
    nbytes = L * read * wb + 2 * h * mc.vocab_size + 2 * T * h + \
        2 * L * mc.kv_size * kvb * (held + T) + 2 * S * mc.vocab_size
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # about four times what exact() is away: 0.0075 (bf16), 0.009 (fp8,
    # also the distance of two implementations that round in other places),
    # 0.007 (Vatunex), 0.005 (experts; near-ties of the router fall either
    # way)
    return {"rel": 2e-2 if case["model"] == "Qwen3-30B-A3B" else 3e-2}


# ------------------------------------------------------------------ exact

def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.to(F64)


def _turn(x, pos, freqs):
    """x [T, heads, D]: entry i turns with entry i + n, n = len(freqs)."""
    a = pos.to(F64)[:, None, None] * freqs
    c, s, n = torch.cos(a), torch.sin(a), freqs.numel()
    u, v = x[..., :n], x[..., n:2 * n]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., 2 * n:]], dim=-1)


def _e4m3(x, per_row=False):
    """Rounded to e4m3; ``per_row``: at a scale that takes the row's largest
    value to 448, as the fp8 mode rounds what enters a projection."""
    if not per_row:
        return x.to(torch.float32).to(F8).to(torch.float32).to(F64)
    s = x.abs().amax(-1, keepdim=True).clamp(min=1e-8) / 448.0
    return _e4m3(x / s) * s


def _attend(q, k, v, first, scale, window=0, one=False):
    """q [n, H, D] at positions first + row; k, v [T, G, D] from position
    0 on."""
    n, H, _ = q.shape
    G = k.shape[1]
    out = torch.empty(n, H, v.shape[2], dtype=F64, device=DEV)
    row = first + torch.arange(n, device=DEV)[:, None]
    col = torch.arange(k.shape[0], device=DEV)[None, :]
    hide = col > row
    if window:
        hide = hide | (col <= row - window)
    for a in range(H):
        g = a // (H // G)
        s = (q[:, a] @ k[:, g].T) * scale
        s.masked_fill_(hide, float("-inf"))
        m = s.amax(1, keepdim=True)
        if one:
            m = m.clamp(min=0.0)
        s.sub_(m).exp_()
        den = s.sum(1, keepdim=True)
        if one:
            den = den + torch.exp(-m)
        out[:, a] = (s @ v[:, g]) / den
    return out


def _plain(tensors):
    """Checkpoint tensors of a layer in 64 bits, e4m3 rows scaled."""
    w = dict(tensors)
    out = {}
    for name, t in w.items():
        if name.endswith("_scale") or ".experts." in name:
            continue
        t = t.to(F64) if t.dtype != F8 else \
            t.float().to(F64) * w[name + "_scale"].to(F64)[:, None]
        out[".".join(name.split(".")[3:])] = t
    return out, w


def _moe(x, router, raw, p, mc):
    probs = torch.softmax(x @ router.T, dim=-1)
    top, ids = probs.topk(mc.num_experts_per_tok, dim=-1)
    top = top / top.sum(-1, keepdim=True)
    out = torch.zeros_like(x)
    for e in range(mc.num_experts):
        r, c = (ids == e).nonzero(as_tuple=True)
        if r.numel() == 0:
            continue
        q = p + f"mlp.experts.{e}."
        g = x[r] @ raw[q + "gate_proj.weight"].to(F64).T
        u = x[r] @ raw[q + "up_proj.weight"].to(F64).T
        y = (torch.nn.functional.silu(g) * u) @ \
            raw[q + "down_proj.weight"].to(F64).T
        out[r] += y * top[r, c][:, None]
    return out


def exact(case, seed):
    with torch.no_grad():
        if case["model"] == "Vatunex":
            return _vatunex_exact(case, seed)
        return _transformer_exact(case, seed)


def _transformer_exact(case, seed):
    mc = _model(case)
    ctx, new, last, prompts = _tokens(case, seed, mc.vocab_size)
    held = list(ctx) + [case["past"]] * len(new)
    # rows of this step: prompts first, then the decoding requests
    spans, row = [], 0
    for i, p in enumerate(prompts):
        spans.append((len(ctx) + i, row, len(p)))
        row += len(p)
    for i in range(len(ctx)):
        spans.append((i, row, 1))
        row += 1
    ids = [t for p in prompts for t in p] + last
    pos = torch.cat([held[s] + torch.arange(n, device=DEV)
                     for s, _, n in spans])
    start = [0]
    for n in held:
        start.append(start[-1] + n)
    enter = (lambda t: _e4m3(t, True)) if case["fp8"] else (lambda t: t)
    outer = dict(_outer_tensors(mc, seed))
    x = outer["model.embed_tokens.weight"][
        torch.tensor(ids, device=DEV)].to(F64)
    H, G, D, eps = mc.num_heads, mc.num_kv_heads, mc.head_dim, mc.rms_norm_eps
    freqs = mc.rope_theta ** (
        -torch.arange(0, D, 2, dtype=F64, device=DEV) / D)
    for i in range(mc.num_layers):
        w, raw = _plain(_layer_tensors(case, mc, seed, i))
        h = enter(_rms(x, w["input_layernorm.weight"], eps))
        q = (h @ w["self_attn.q_proj.weight"].T).view(-1, H, D)
        k = (h @ w["self_attn.k_proj.weight"].T).view(-1, G, D)
        v = (h @ w["self_attn.v_proj.weight"].T).view(-1, G, D)
        q = _turn(_rms(q, w["self_attn.q_norm.weight"], eps), pos, freqs)
        k = _turn(_rms(k, w["self_attn.k_norm.weight"], eps), pos, freqs)
        if case["fp8_kv"]:
            k, v = _e4m3(k), _e4m3(v)
        if start[-1]:
            old = [_context(mc, seed, i, n, start[-1]).to(F64)
                   .view(-1, G, D) for n in "kv"]
            if case["fp8_kv"]:
                old = [_e4m3(t) for t in old]
        a = torch.empty_like(q)
        for s, r, n in spans:
            ks, vs = k[r:r + n], v[r:r + n]
            if held[s]:
                part = slice(start[s], start[s + 1])
                ks = torch.cat([old[0][part], ks])
                vs = torch.cat([old[1][part], vs])
            a[r:r + n] = _attend(q[r:r + n], ks, vs, held[s], D ** -0.5)
        x = x + enter(a.reshape(-1, H * D)) @ w["self_attn.o_proj.weight"].T
        h = enter(_rms(x, w["post_attention_layernorm.weight"], eps))
        if mc.is_moe:
            x = x + _moe(h, w["mlp.gate.weight"], raw,
                         f"model.layers.{i}.", mc)
        else:
            y = torch.nn.functional.silu(h @ w["mlp.gate_proj.weight"].T) * \
                (h @ w["mlp.up_proj.weight"].T)
            x = x + enter(y) @ w["mlp.down_proj.weight"].T
    rows = [r + n - 1 for _, r, n in spans]
    x = _rms(x[rows], outer["model.norm.weight"], eps)
    return x @ outer["lm_head.weight"].to(F64).T


# ---------------------------------------------------------------- Vatunex

def _vatunex():
    width, heads, dim = 2048, 16, 128
    dense = {"kind": "dense", "ff": 3 * width}
    latent = {"heads": heads, "dim": 96, "rot_dim": 32, "vdim": dim,
              "kv_rank": 256, "q_rank": 3 * width // 8,
              "scale": dim ** -0.5, "mask": {"size": 1024},
              "rot": {"base": 1e6, "dims": 32}}
    attention = {"heads": heads, "kv_heads": heads // 4, "dim": dim,
                 "vdim": dim, "scale": dim ** -0.5, "v_mix": True,
                 "rot": {"base": 5e5, "dims": dim,
                         "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0,
                                     "original": 8192}}}
    scan = {"inner": 2 * width, "state": 16, "conv": 4,
            "dt_rank": width // 16}
    return {"architecture": "Vatunex", "vocab": 32000, "width": width,
            "norm": {"eps": 1e-5},
            "layers": [
                {"type": "latent_attention", "mixer": latent, "mlp": dense},
                {"type": "attention", "mixer": attention, "mlp": dense},
                {"type": "mamba1", "mixer": scan, "mlp": dense},
                {"type": "attention", "mixer": attention, "mlp": dense}]}


def _vatunex_tensors(seed):
    """Checkpoint tensors, matrices in bf16 and small ones in fp32."""
    raw = _vatunex()
    W = raw["width"]

    def mat(name, rows, cols):
        return name, _normal(seed, name, (rows, cols))

    def vec(name, n, lo, hi):
        return name, _uniform(seed, name, (n,), lo, hi)

    yield mat("embed", raw["vocab"], W)
    yield mat("head", raw["vocab"], W)
    yield vec("final.norm", W, -0.2, 0.2)
    for i, layer in enumerate(raw["layers"]):
        p, m = f"l{i}.mix.", layer["mixer"]
        for n in ("1", "1b", "2", "2b"):
            yield vec(f"l{i}.norm{n}", W, -0.5, 0.5)
        yield mat(f"l{i}.mlp.up", layer["mlp"]["ff"], W)
        yield mat(f"l{i}.mlp.down", W, layer["mlp"]["ff"])
        if layer["type"] == "mamba1":
            n, s, r = m["inner"], m["state"], m["dt_rank"]
            yield mat(p + "in", 2 * n, W)
            yield p + "conv", _uniform(seed, p + "conv", (n, m["conv"]),
                                       -0.6, 0.6)
            yield vec(p + "conv.b", n, -0.2, 0.2)
            yield mat(p + "x", r + 2 * s, n)
            yield mat(p + "dt", n, r)
            yield vec(p + "dt.b", n, -4.0, 0.0)
            yield p + "A_log", _uniform(seed, p + "A_log", (n, s), -1.0, 2.0)
            yield vec(p + "D", n, 0.5, 1.5)
            yield mat(p + "o", W, n)
            continue
        H, D, V = m["heads"], m["dim"], m["vdim"]
        yield mat(p + "o", W, H * V)
        if layer["type"] == "latent_attention":
            R, Q, N = m["rot_dim"], m["q_rank"], m["kv_rank"]
            yield mat(p + "dq", Q, W)
            yield vec(p + "dq.norm", Q, 0.5, 1.5)
            yield mat(p + "uq", H * (D + R), Q)
            yield mat(p + "dkv", N + R, W)
            yield vec(p + "dkv.norm", N, 0.5, 1.5)
            yield mat(p + "uk", H * D, N)
            yield mat(p + "uv", H * V, N)
            continue
        G = m["kv_heads"]
        for n, rows in (("q", H * D), ("k", G * D), ("v", G * V)):
            yield mat(p + n, rows, W)
            yield vec(p + n + ".b", rows, -0.3, 0.3)
        yield vec(p + "o.b", W, -0.3, 0.3)
        yield vec(p + "q.norm", D, 0.5, 1.5)
        yield vec(p + "k.norm", D, 0.5, 1.5)
        yield p + "vmix", _uniform(seed, p + "vmix", (), 0.2, 0.8)


def _vatunex_work(case, new):
    raw, steps = _vatunex(), case["steps"]
    W, V = raw["width"], raw["vocab"]
    params, flops, state, old = 0, 0, 0, 0
    T = sum(new) + steps * len(new)
    for layer in raw["layers"]:
        m, ff = layer["mixer"], layer["mlp"]["ff"]
        params += 2 * W * ff
        if layer["type"] == "mamba1":
            n, s, r = m["inner"], m["state"], m["dt_rank"]
            params += 3 * W * n + n * (r + 2 * s) + r * n
            flops += T * n * (6 * s + 2 * m["conv"])
            # the state is written after the prompt, read and written in
            # every decode step
            state += 4 * n * s * len(new) * (1 + 2 * steps)
            continue
        H, D = m["heads"], m["dim"]
        if layer["type"] == "latent_attention":
            params += W * (m["q_rank"] + m["kv_rank"] + m["rot_dim"]) + \
                H * (m["q_rank"] * (D + m["rot_dim"]) +
                     m["kv_rank"] * (D + m["vdim"]) + W * m["vdim"])
            D += m["rot_dim"]
            row = m["kv_rank"] + m["rot_dim"]
        else:
            G = m["kv_heads"]
            params += W * (H * D + G * (D + m["vdim"]) + H * m["vdim"])
            row = G * (D + m["vdim"])
        w = (m.get("mask") or {}).get("size") or 10 ** 9
        pairs = sum(sum(min(t + 1, w) for t in range(n + steps))
                    for n in new)
        flops += 2 * H * (D + m["vdim"]) * pairs
        old += 2 * row * sum(min(n + t + 1, w) for n in new
                             for t in range(steps)) + 2 * row * T
    S = len(new) * (1 + steps)
    flops += 2 * params * T + 2 * S * W * V
    nbytes = (1 + steps) * 2 * (params + W * V) + 2 * T * W + 4 * S * V + \
        state + old
    return {"bytes": nbytes, "flops": flops}


def _stretched(rot):
    n = rot["dims"] // 2
    f = rot["base"] ** (-torch.arange(n, dtype=F64, device=DEV) / n)
    sc = rot.get("scaling")
    if sc:
        turns = sc["original"] * f / (2.0 * math.pi)
        keep = ((turns - sc["low"]) / (sc["high"] - sc["low"])).clamp(0, 1)
        f = keep * f + (1.0 - keep) * f / sc["factor"]
    return f


def _vatunex_scan(h, w, m):
    n, N, R = m["inner"], m["state"], m["dt_rank"]
    xz = h @ w["in"].T
    x, z = xz[:, :n], xz[:, n:]
    taps = m["conv"]
    pad = torch.cat([torch.zeros(taps - 1, n, dtype=F64, device=DEV), x])
    x = sum(pad[j:j + x.shape[0]] * w["conv"][:, j] for j in range(taps))
    x = torch.nn.functional.silu(x + w["conv.b"])
    p = x @ w["x"].T
    dt = torch.nn.functional.softplus(p[:, :R] @ w["dt"].T + w["dt.b"])
    A, B, C = -torch.exp(w["A_log"]), p[:, R:R + N], p[:, R + N:]
    S = torch.zeros_like(A)
    y = torch.empty_like(x)
    dx = dt * x
    for t in range(x.shape[0]):
        S = torch.exp(dt[t][:, None] * A) * S + dx[t][:, None] * B[t]
        y[t] = S @ C[t]
    return ((y + w["D"] * x) * torch.nn.functional.silu(z)) @ w["o"].T


def _vatunex_exact(case, seed):
    raw = _vatunex()
    eps, steps = raw["norm"]["eps"], case["steps"]
    W = {k: t.to(F64) for k, t in _vatunex_tensors(seed)}
    _, new, _, prompts = _tokens(case, seed, raw["vocab"])
    rows = []
    for n, p in zip(new, prompts):
        x = W["embed"][torch.tensor(p, device=DEV)]
        pos = torch.arange(x.shape[0], device=DEV)
        v_first = None
        for i, layer in enumerate(raw["layers"]):
            pre, m = f"l{i}.mix.", layer["mixer"]
            w = {k[len(pre):]: t for k, t in W.items() if k.startswith(pre)}
            h = _rms(x, 1.0 + W[f"l{i}.norm1"], eps)
            if layer["type"] == "mamba1":
                y = _vatunex_scan(h, w, m)
            else:
                H, D = m["heads"], m["dim"]
                freqs = _stretched(m["rot"])
                if layer["type"] == "latent_attention":
                    c = h @ w["dkv"].T
                    k_rot = c[:, None, m["kv_rank"]:]
                    c = _rms(c[:, :m["kv_rank"]], w["dkv.norm"], eps)
                    q = _rms(h @ w["dq"].T, w["dq.norm"], eps) @ w["uq"].T
                    q = q.view(-1, H, D + m["rot_dim"])
                    q = torch.cat([q[..., :D],
                                   _turn(q[..., D:], pos, freqs)], dim=-1)
                    k = torch.cat(
                        [(c @ w["uk"].T).view(-1, H, D),
                         _turn(k_rot, pos, freqs).expand(-1, H, -1)], dim=-1)
                    v = (c @ w["uv"].T).view(-1, H, m["vdim"])
                    y = _attend(q, k, v, 0, m["scale"], m["mask"]["size"])
                    y = y.reshape(len(p), -1) @ w["o"].T
                else:
                    G = m["kv_heads"]
                    q, k, v = (h @ w[t].T + w[t + ".b"] for t in "qkv")
                    if v_first is None:
                        v_first = v
                    else:
                        v = (1.0 - w["vmix"]) * v + w["vmix"] * v_first
                    q = _rms(q.view(-1, H, D), w["q.norm"], eps)
                    k = _rms(k.view(-1, G, D), w["k.norm"], eps)
                    y = _attend(_turn(q, pos, freqs), _turn(k, pos, freqs),
                                v.view(-1, G, m["vdim"]), 0, m["scale"],
                                one=True)
                    y = y.reshape(len(p), -1) @ w["o"].T + w["o.b"]
            x = x + _rms(y, 1.0 + W[f"l{i}.norm1b"], eps)
            h = _rms(x, 1.0 + W[f"l{i}.norm2"], eps)
            y = torch.nn.functional.gelu(h @ W[f"l{i}.mlp.up"].T,
                                         approximate="tanh")
            x = x + _rms(y @ W[f"l{i}.mlp.down"].T,
                         1.0 + W[f"l{i}.norm2b"], eps)
        x = _rms(x[n - 1:], 1.0 + W["final.norm"], eps)
        rows.append(x @ W["head"].T)
    # one output per step, a row per request
    return [torch.stack([r[t] for r in rows]) for t in range(steps + 1)]
