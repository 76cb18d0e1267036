"""Work that users have this framework do, as cases that can be timed.

Language models are served by LLMEngine: one pass is one model step, given to
LLMEngine.extend() as token ids, with logits as its result. It is the step
that serving takes as well; sampling comes after it. The embedding model and
the image model are called as their serving instances call them.

Weights, cached keys and values and token ids are random, made from the seed.
The spread of the weights is the usual one for a start of training, but a
token's embedding outweighs what a single layer adds to it, as the sum of all
layers before does in trained models: else roundings are blown up from layer
to layer. Sizes are those of the presets, of bench.py and of the serving limits.

A case of a language model says how many sequences go on by one token
("rows", their lengths in tokens from "row_lo" to "row_hi", the new one
included) and how many get a prompt portion ("portions" of "new_lo" to
"new_hi" tokens, behind "cached" tokens that are in the cache already).
"""
import math
import random
import zlib
from dataclasses import replace

import torch

from helix_amd.engine.engine import (EngineConfig, LLMEngine, Sequence,
                                     SeqStatus)
from helix_amd.engine.sampling_params import SamplingParams
from helix_amd.models.bert import BERT_PRESETS, BertEmbeddingModel
from helix_amd.models.dit import DIT_PRESETS, DiTModel
from helix_amd.models.llama import PRESETS, LlamaForCausalLM
from helix_amd.ops import make_cos_sin_cache

DEV = "cuda"
PAGE = 16                 # tokens of a cache page, the engine's default
STD = 0.02                # of random weights


def _lm(name, model, rows=0, row_lo=0, row_hi=0, portions=0, new_lo=0,
        new_hi=0, cached=0, want="last", layers=0, weights="bf16",
        cache="bf16"):
    return {"name": name, "do": "lm", "model": model, "rows": rows,
            "row_lo": row_lo, "row_hi": row_hi, "portions": portions,
            "new_lo": new_lo, "new_hi": new_hi, "cached": cached,
            "want": want, "layers": layers, "weights": weights,
            "cache": cache}


def listed():
    return [
        # one user's chat reply, token by token: latency
        _lm("reply to one", "llama3-8b", 1, 777, 777),
        # a few users of the model with a sliding window, some beyond it
        _lm("replies to eight", "mistral-7b", 8, 300, 6000),
        # a busy server with long conversations
        _lm("replies to sixty-one", "llama3-8b", 61, 1000, 4096),
        # the largest batch that is captured as a graph: bench.py's step
        _lm("replies to 512", "llama3-8b", 512, 513, 640),
        # long documents with the 8-bit cache
        _lm("replies, 8-bit cache", "llama3.1-8b", 24, 4000, 16000,
            cache="fp8"),
        # 8-bit weights and activations; four layers, because a rounding to
        # 3 bits that falls the other way is carried on by every layer
        _lm("replies, 8-bit weights", "llama3-8b", 32, 200, 2000, layers=4,
            weights="fp8"),
        # a question of one line, scored at every place (log-probabilities)
        _lm("short prompt, scored", "llama3-8b", portions=1, new_lo=37,
            new_hi=37, want="all"),
        # admission of many prompts in one step of 16k tokens, as in bench.py
        _lm("batch of prompts", "llama3-8b", portions=31, new_lo=400,
            new_hi=620),
        # one long document
        _lm("long prompt", "llama3.1-8b", portions=1, new_lo=8192,
            new_hi=8192),
        # the next portion of a conversation behind a cached prefix, beside
        # the replies of a mixed step
        _lm("portion beside replies", "mistral-7b", 40, 100, 3000, 1, 1500,
            1500, cached=5001),
        # documents on their way into the vector store
        {"name": "embeddings", "do": "embed", "model": "bge-base",
         "texts": 64, "lo": 20, "hi": 500},
        # one step of image generation
        {"name": "image step", "do": "image", "model": "flux-lite",
         "images": 8},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo),
                                                      math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["replies", "replies", "replies", "prompts", "prompts",
                       "mixed", "embed", "image"])
    model = rng.choice(["llama3-8b", "mistral-7b"])
    if kind == "embed":
        return {"do": "embed",
                "model": rng.choice(["bge-base", "bge-base", "bge-large"]),
                "texts": _log(rng, 1, 64), "lo": _log(rng, 4, 100),
                "hi": rng.randint(101, 511)}
    if kind == "image":
        return {"do": "image", "model": "flux-lite",
                "images": rng.randint(1, 8)}
    case = _lm("", model)
    del case["name"]
    if kind == "replies":
        rows = _log(rng, 1, 512)
        # about as much cache as the largest listed cases at most
        case.update(rows=rows, row_lo=_log(rng, 20, 400),
                    row_hi=_log(rng, 401, min(8000, 160000 // rows + 401)))
        if rng.random() < 0.2 and rows <= 64:
            case.update(model="llama3.1-8b", cache="fp8")
        elif rng.random() < 0.15 and rows <= 64:
            case.update(model="llama3-8b", weights="fp8", layers=4)
    elif kind == "prompts":
        n = _log(rng, 1, 31)
        top = min(8000, 16000 // n)
        case.update(portions=n, new_lo=_log(rng, 5, top // 2),
                    new_hi=rng.randint(top // 2 + 1, top))
        if case["new_hi"] * n <= 64 and rng.random() < 0.5:
            case.update(want="all")
    else:
        case.update(rows=_log(rng, 2, 64), row_lo=_log(rng, 20, 300),
                    row_hi=_log(rng, 301, 4000),
                    portions=rng.randint(1, 2), new_lo=_log(rng, 17, 300),
                    new_hi=_log(rng, 301, 2000),
                    cached=rng.choice([0, _log(rng, 16, 5000)]))
    return case


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _key(case, *more):
    text = repr(sorted((k, v) for k, v in case.items() if k != "name"))
    return zlib.crc32((text + repr(more)).encode())


def _spread(case, what, n, lo, hi):
    """n lengths in [lo, hi], the same for every seed; lo and hi are met."""
    rng = random.Random(_key(case, what))
    out = [rng.randint(lo, hi) for _ in range(n)]
    if n:
        out[0] = hi
    if n > 1:
        out[-1] = lo
    return out


def _spans(case):
    """(tokens before, tokens new) of every sequence."""
    rows = _spread(case, "rows", case["rows"], case["row_lo"], case["row_hi"])
    new = _spread(case, "new", case["portions"], case["new_lo"],
                  case["new_hi"])
    return [(n - 1, 1) for n in rows] + [(case["cached"], n) for n in new]


def _gen(seed, *what):
    return torch.Generator(device=DEV).manual_seed(
        zlib.crc32(repr(what).encode()) * 65537 + seed)


def _normal(t, seed, std, *what):
    return t.normal_(0.0, std, generator=_gen(seed, *what))


def _config(case):
    cfg = PRESETS[case["model"]]
    return replace(cfg, num_layers=case["layers"]) if case["layers"] else cfg


def _fill(model, seed, layers=0):
    for name, p in model.named_parameters():
        _weight(p.data, name, seed, layers)


def _weight(t, name, seed, layers=0):
    """Random weights; those of norms around 1. layers: depth of a language
    model, whose layers' last projections share the growth of the sum."""
    std = STD
    if name.endswith(("norm_w", "ln_w")):
        return _normal(t, seed, 0.1, name).add_(1.0)
    if layers and name.startswith("embed"):
        std = 4.0
    elif layers and name.endswith(("o_proj.weight", "down_proj.weight")):
        std = STD / math.sqrt(2 * layers)
    return _normal(t, seed, std, name)


def _construct(make):
    """A model on the GPU in bf16, without initialising it on the host."""
    kind = torch.get_default_dtype()
    torch.set_default_dtype(torch.bfloat16)
    try:
        with torch.device(DEV):
            return make()
    finally:
        torch.set_default_dtype(kind)


def _kv_std(cfg):
    """Spread of a projection of a normed row."""
    return STD * math.sqrt(cfg.hidden_size)


def _tables(case, seed):
    """Pages of every sequence, in no order, as after some time of serving;
    and the number of pages."""
    need = [-(-(a + b) // PAGE) for a, b in _spans(case)]
    pages = list(range(sum(need)))
    random.Random(seed).shuffle(pages)
    out, at = [], 0
    for n in need:
        out.append(pages[at:at + n])
        at += n
    return out, at


def _cached(t, cfg, seed, layer, which, fp8):
    """The pages of one layer's keys or values."""
    if fp8:
        b = torch.empty(t.shape, dtype=torch.bfloat16, device=DEV)
        _normal(b, seed, _kv_std(cfg), "cache", layer, which)
        return t.copy_(b.to(torch.float8_e4m3fn).view(torch.uint8))
    return _normal(t, seed, _kv_std(cfg), "cache", layer, which)


def _ids(case, cfg, seed):
    rng = random.Random(seed * 7 + 3)
    return [[rng.randrange(cfg.vocab_size) for _ in range(n)]
            for _, n in _spans(case)]


def prepare(case, seed):
    return {"lm": _prepare_lm, "embed": _prepare_embed,
            "image": _prepare_image}[case["do"]](case, seed)


def _prepare_lm(case, seed):
    cfg = _config(case)
    spans = _spans(case)
    tables, pages = _tables(case, seed)
    model = _construct(lambda: LlamaForCausalLM(cfg))
    model.cos_sin = make_cos_sin_cache(
        cfg.head_dim, cfg.max_position, cfg.rope_base,
        rope_scaling=cfg.rope_scaling or None).to(DEV)
    _fill(model, seed, cfg.num_layers)
    eng = LLMEngine(EngineConfig(
        model=case["model"], max_num_seqs=max(64, len(spans)),
        max_model_len=min(cfg.max_position, 16384),
        max_prefill_tokens=16384, kv_cache_blocks=pages, eos_token_id=-1,
        quantization="fp8" if case["weights"] == "fp8" else None,
        kv_cache_dtype=case["cache"], mixed_steps=True), DEV, model=model)
    eng.kv.allocator.allocate(pages)
    for i, (k, v) in enumerate(eng.kv.caches):
        if any(before for before, _ in spans):
            _cached(k, cfg, seed, i, "k", case["cache"] == "fp8")
            _cached(v, cfg, seed, i, "v", case["cache"] == "fp8")
    ids = _ids(case, cfg, seed)
    entries, keep = [], {}
    for n, (before, new) in enumerate(spans):
        sid = "s%d" % n
        eng.seqs[sid] = Sequence(sid, [1] * before, SamplingParams(),
                                 status=SeqStatus.RUNNING,
                                 block_table=tables[n])
        keep[sid] = before
        want = list(range(new)) if case["want"] == "all" else [new - 1]
        entries.append((sid, ids[n], want))
    return {"run": _run_lm, "engine": eng, "entries": entries, "keep": keep}


def _run_lm(s):
    logits = s["engine"].extend(s["entries"])
    # the tokens are taken back, so that the next pass is the same step
    for sid, n in s["keep"].items():
        del s["engine"].seqs[sid].prompt_ids[n:]
    return logits


def _prepare_embed(case, seed):
    cfg = BERT_PRESETS[case["model"]]
    model = _construct(lambda: BertEmbeddingModel(cfg))
    _fill(model, seed)
    lens = _spread(case, "texts", case["texts"], case["lo"], case["hi"])
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    return {"run": _run_embed, "model": model, "longest": max(lens),
            "ids": _text_ids(cfg, cu[-1], seed),
            "cu": torch.tensor(cu, dtype=torch.int32, device=DEV)}


def _text_ids(cfg, n, seed):
    return torch.randint(0, cfg.vocab_size, (n,), device=DEV,
                         generator=_gen(seed, "ids"))


def _run_embed(s):
    return s["model"](s["ids"], s["cu"], s["longest"])


def _image_inputs(cfg, n, seed):
    lat = torch.empty(n, cfg.latent_ch, cfg.latent_size, cfg.latent_size,
                      dtype=torch.bfloat16, device=DEV)
    ids = torch.randint(0, cfg.vocab_size, (n, cfg.text_len), device=DEV,
                        generator=_gen(seed, "ids"))
    return (_normal(lat, seed, 1.0, "latents"),
            torch.full((n,), 0.75, device=DEV), ids)


def _prepare_image(case, seed):
    cfg = DIT_PRESETS[case["model"]]
    model = _construct(lambda: DiTModel(cfg))
    _fill(model, seed)
    return {"run": _run_image, "model": model,
            "inputs": _image_inputs(cfg, case["images"], seed)}


def _run_image(s):
    with torch.inference_mode():
        return s["model"](*s["inputs"])


def run(state):
    return state["run"](state)


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    if case["do"] == "lm":
        return _work_lm(case)
    if case["do"] == "embed":
        cfg = BERT_PRESETS[case["model"]]
        lens = _spread(case, "texts", case["texts"], case["lo"], case["hi"])
        T, h = sum(lens), cfg.hidden_size
        layer = 4 * h * h + 2 * h * cfg.intermediate_size
        flops = cfg.num_layers * (2 * T * layer
                                  + 4 * h * sum(n * n for n in lens))
        return {"flops": flops, "bytes": 2 * cfg.num_layers * layer
                + 2 * 2 * T * h + 8 * T + 4 * len(lens) * h}
    cfg = DIT_PRESETS[case["model"]]
    n, L, h = case["images"], cfg.seq_len, cfg.hidden
    lat = n * cfg.latent_ch * cfg.latent_size ** 2
    blocks = 12 * h * h
    mods = cfg.depth * 6 * h * h + 3 * h * h + cfg.time_dim * h
    flops = cfg.depth * (2 * n * L * blocks + 4 * n * L * L * h) \
        + 2 * n * mods + 2 * n * L * 2 * h * cfg.patch_dim
    return {"flops": flops, "bytes": 2 * (cfg.depth * blocks + mods)
            + 2 * lat + 4 * lat + 2 * n * cfg.text_len * h}


def _work_lm(case):
    cfg = _config(case)
    spans = _spans(case)
    T = sum(n for _, n in spans)
    outs = T if case["want"] == "all" else len(spans)
    layer = cfg.num_weights()[1] // cfg.num_layers
    head = cfg.vocab_size * cfg.hidden_size
    window = cfg.sliding_window or 1 << 30
    seen = sum(min(a + i + 1, window) for a, n in spans for i in range(n))
    read = sum(min(a, window - 1) for a, _ in spans)
    wide = 1 if case["weights"] == "fp8" else 2
    elem = 1 if case["cache"] == "fp8" else 2
    flops = 2 * T * layer * cfg.num_layers + 2 * outs * head \
        + cfg.num_layers * 4 * cfg.q_size * seen
    bytes_ = wide * layer * cfg.num_layers + 2 * head \
        + cfg.num_layers * 2 * cfg.kv_size * elem * (read + T) \
        + 2 * T * cfg.hidden_size + 2 * outs * cfg.vocab_size
    return {"flops": flops, "bytes": bytes_}


# ---------------------------------------------------------------------------
# How exact a result is
# ---------------------------------------------------------------------------

def tolerance(case):
    """bf16 from layer to layer: another order of the sums in the projections
    changes logits by 0.009 to 0.012 (largest single difference 0.06 of the
    root mean square); 64 bits are 0.011 to 0.022 away in all cases."""
    return {"rel": 0.03, "max": 0.25}


def exact(case, seed):
    with torch.inference_mode():
        return {"lm": _exact_lm, "embed": _exact_embed,
                "image": _exact_image}[case["do"]](case, seed)


def _w(name, shape, seed, layers=0):
    t = torch.empty(shape, dtype=torch.bfloat16, device=DEV)
    return _weight(t, name, seed, layers).double()


def _rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _e4m3(x):
    """Rounded to 8 bits with one scale per row."""
    s = x.float().abs().amax(-1, keepdim=True).clamp(min=1e-8) / 448.0
    return (x.float() / s).to(torch.float8_e4m3fn).double() * s.double()


def _frequencies(cfg):
    half = cfg.head_dim // 2
    f = cfg.rope_base ** (-torch.arange(half, dtype=torch.float64,
                                        device=DEV) / half)
    r = cfg.rope_scaling
    if r:
        turns = r["original_max_position_embeddings"] * f / (2 * math.pi)
        mix = ((turns - r["low_freq_factor"])
               / (r["high_freq_factor"] - r["low_freq_factor"])).clamp(0, 1)
        f = f / r["factor"] * (1 - mix) + f * mix
    return f


def _turn(x, pos, freq):
    """x [T, H, D], first and second half of a head are the pairs."""
    a = pos[:, None, None].double() * freq
    u, v = x.chunk(2, -1)
    return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()],
                     -1)


def _attend(q, k, v, before, window, causal=True):
    """q [n, H, D] at positions before.., k and v [before + n, G, D]."""
    n, H, D = q.shape
    L, G = k.shape[:2]
    kt = k.permute(1, 2, 0).contiguous()
    vt = v.permute(1, 0, 2).contiguous()
    out = torch.empty_like(q)
    at = torch.arange(L, device=DEV)
    step = max(1, (1 << 28) // (H * L))
    for a in range(0, n, step):
        b = min(n, a + step)
        x = q[a:b].view(b - a, G, H // G, D).permute(1, 2, 0, 3) \
            .reshape(G, -1, D)
        s = ((x @ kt) * D ** -0.5).view(G, H // G, b - a, L)
        if causal:
            p = torch.arange(before + a, before + b, device=DEV)[:, None]
            hide = at > p
            if window:
                hide |= at <= p - window
            s.masked_fill_(hide, -math.inf)
        s = torch.softmax(s, -1).view(G, -1, L)
        out[a:b] = (s @ vt).view(G, H // G, b - a, D).permute(2, 0, 1, 3) \
            .reshape(b - a, H, D)
    return out


def _exact_lm(case, seed):
    cfg = _config(case)
    spans = _spans(case)
    tables, pages = _tables(case, seed)
    h, D, G = cfg.hidden_size, cfg.head_dim, cfg.num_kv_heads
    q_size, kv, ff = cfg.q_size, cfg.kv_size, cfg.intermediate_size
    fp8, fp8_kv = case["weights"] == "fp8", case["cache"] == "fp8"
    ids = torch.tensor([t for s in _ids(case, cfg, seed) for t in s],
                       device=DEV)
    pos = torch.tensor([a + i for a, n in spans for i in range(n)],
                       device=DEV)
    at = [torch.tensor([t[p // PAGE] * PAGE + p % PAGE for p in range(a)],
                       device=DEV) for t, (a, _) in zip(tables, spans)]
    freq = _frequencies(cfg)

    def linear(x, name, shape):
        w = _w(name, shape, seed, cfg.num_layers)
        if fp8:
            x, w = _e4m3(x), _e4m3(w)
        return x @ w.t()

    def pages_of(layer, which):
        t = torch.empty(pages, G, PAGE, D, device=DEV,
                        dtype=torch.uint8 if fp8_kv else torch.bfloat16)
        _cached(t, cfg, seed, layer, which, fp8_kv)
        t = t.view(torch.float8_e4m3fn).bfloat16() if fp8_kv else t
        return t.transpose(1, 2).reshape(pages * PAGE, G, D)

    x = _w("embed_tokens.weight", (cfg.vocab_size, h), seed, 1)[ids]
    for i in range(cfg.num_layers):
        n = "layers.%d." % i
        y = _rms(x, _w(n + "input_norm_w", (h,), seed), cfg.rms_norm_eps)
        y = linear(y, n + "attn.qkv_proj.weight", (q_size + 2 * kv, h))
        q, k, v = y.split([q_size, kv, kv], -1)
        q = _turn(q.reshape(-1, cfg.num_heads, D), pos, freq)
        k = _turn(k.reshape(-1, G, D), pos, freq)
        v = v.reshape(-1, G, D)
        if fp8_kv:
            k, v = (t.to(torch.float8_e4m3fn).double() for t in (k, v))
        o = torch.empty_like(q)
        if any(a for a, _ in spans):
            ks, vs = pages_of(i, "k"), pages_of(i, "v")
        r = 0
        for slots, (a, new) in zip(at, spans):
            s = slice(r, r + new)
            r += new
            if a:
                ka = torch.cat([ks[slots].double(), k[s]])
                va = torch.cat([vs[slots].double(), v[s]])
            else:
                ka, va = k[s], v[s]
            o[s] = _attend(q[s], ka, va, a, cfg.sliding_window)
        x = x + linear(o.reshape(-1, q_size), n + "attn.o_proj.weight",
                       (h, q_size))
        y = _rms(x, _w(n + "post_norm_w", (h,), seed), cfg.rms_norm_eps)
        g, u = linear(y, n + "mlp.gate_up_proj.weight",
                      (2 * ff, h)).chunk(2, -1)
        x = x + linear(torch.nn.functional.silu(g) * u,
                       n + "mlp.down_proj.weight", (h, ff))
    ends = torch.tensor([n for _, n in spans], device=DEV).cumsum(0) - 1
    if case["want"] != "all":
        x = x[ends]
    x = _rms(x, _w("final_norm_w", (h,), seed), cfg.rms_norm_eps)
    return x @ _w("lm_head.weight", (cfg.vocab_size, h), seed).t()


def _norm(x, eps, w=1.0, b=0.0):
    x = x - x.mean(-1, keepdim=True)
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w + b


def _gelu(x):
    return torch.nn.functional.gelu(x, approximate="tanh")


def _heads(qkv, heads):
    return (t.reshape(t.shape[0], heads, -1) for t in qkv.chunk(3, -1))


def _exact_embed(case, seed):
    cfg = BERT_PRESETS[case["model"]]
    lens = _spread(case, "texts", case["texts"], case["lo"], case["hi"])
    h, ff, eps = cfg.hidden_size, cfg.intermediate_size, cfg.layer_norm_eps
    ids = _text_ids(cfg, sum(lens), seed)
    pos = torch.cat([torch.arange(n, device=DEV) for n in lens])
    w = lambda name, *shape: _w(name, shape, seed)  # noqa: E731
    x = w("word_emb.weight", cfg.vocab_size, h)[ids] \
        + w("pos_emb.weight", cfg.max_position, h)[pos]
    x = _norm(x, eps, w("emb_ln_w", h), w("emb_ln_b", h))
    for i in range(cfg.num_layers):
        n = "layers.%d." % i
        qkv = x @ w(n + "qkv_w", 3 * h, h).t() + w(n + "qkv_b", 3 * h)
        q, k, v = _heads(qkv, cfg.num_heads)
        o, r = torch.empty_like(q), 0
        for t in lens:
            s = slice(r, r + t)
            o[s] = _attend(q[s], k[s], v[s], 0, 0, causal=False)
            r += t
        a = o.reshape(-1, h) @ w(n + "attn_out_w", h, h).t() \
            + w(n + "attn_out_b", h)
        x = _norm(x + a, eps, w(n + "attn_ln_w", h), w(n + "attn_ln_b", h))
        m = _gelu(x @ w(n + "up_w", ff, h).t() + w(n + "up_b", ff))
        m = m @ w(n + "down_w", h, ff).t() + w(n + "down_b", h)
        x = _norm(x + m, eps, w(n + "out_ln_w", h), w(n + "out_ln_b", h))
    first = torch.tensor([0] + lens[:-1], device=DEV).cumsum(0)
    return torch.nn.functional.normalize(x[first], dim=-1)


def _exact_image(case, seed):
    cfg = DIT_PRESETS[case["model"]]
    B, p, h, L = case["images"], cfg.patch, cfg.hidden, cfg.seq_len
    lat, t, ids = _image_inputs(cfg, B, seed)
    w = lambda name, *shape: _w(name, shape, seed)  # noqa: E731
    g, C, P = cfg.latent_size // p, cfg.latent_ch, cfg.num_patches
    rows = lat.double().view(B, C, g, p, g, p).permute(0, 2, 4, 1, 3, 5) \
        .reshape(B * P, cfg.patch_dim)
    pad = -(-cfg.patch_dim // 64) * 64
    img = rows @ w("in_w", h, pad)[:, :cfg.patch_dim].t() + w("in_b", h)
    tx = w("txt_emb.weight", cfg.vocab_size, h)[ids]
    x = torch.cat([tx, img.view(B, P, h)], 1) + w("pos_emb.weight", L, h)
    half = cfg.time_dim // 2
    f = 10000.0 ** (-torch.arange(half, dtype=torch.float64, device=DEV)
                    / half)
    a = t.double()[:, None] * 1000.0 * f
    c = _gelu(torch.cat([a.cos(), a.sin()], -1)
              @ w("t_w1", h, cfg.time_dim).t() + w("t_b1", h))
    c = c @ w("t_w2", h, h).t() + w("t_b2", h) + tx.mean(1)
    for i in range(cfg.depth):
        n = "blocks.%d." % i
        mod = (c @ w(n + "mod_w", 6 * h, h).t() + w(n + "mod_b", 6 * h))
        sa, ca, ga, sm, cm, gm = mod[:, None].chunk(6, -1)
        y = _norm(x, cfg.eps) * (1 + ca) + sa
        qkv = y @ w(n + "qkv_w", 3 * h, h).t() + w(n + "qkv_b", 3 * h)
        o = torch.stack([_attend(*_heads(r, cfg.heads), 0, 0, causal=False)
                         for r in qkv]).view(B, L, h)
        x = x + ga * (o @ w(n + "out_w", h, h).t() + w(n + "out_b", h))
        y = _norm(x, cfg.eps) * (1 + cm) + sm
        y = _gelu(y @ w(n + "up_w", 4 * h, h).t() + w(n + "up_b", 4 * h))
        x = x + gm * (y @ w(n + "down_w", h, 4 * h).t()
                      + w(n + "down_b", h))
    shift, scale = (c @ w("fin_mod_w", 2 * h, h).t()
                    + w("fin_mod_b", 2 * h))[:, None].chunk(2, -1)
    y = _norm(x, cfg.eps) * (1 + scale) + shift
    y = (y @ w("fin_w", cfg.patch_dim, h).t() + w("fin_b", cfg.patch_dim))
    return y[:, L - P:].reshape(B, g, g, C, p, p) \
        .permute(0, 3, 1, 4, 2, 5).reshape(B, C, g * p, g * p)
