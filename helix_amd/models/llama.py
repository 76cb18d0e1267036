"""Llama-family decoder (Llama-3 8B/70B, Mistral-7B) on helix_amd CDNA4 ops.

Replaces the model execution the reference delegates to vLLM containers
(SURVEY.md §2.8): hand-written HIP kernels for RMSNorm/RoPE/attention/
activation and projections (ops.linear; the library's GEMM where it is the
faster one, vocabularies of few rows among them); paged KV.

Tensor-parallel sharding (RCCL over xGMI) is applied by
helix_amd.parallel when tp_size > 1: column-parallel QKV/gate_up,
row-parallel o_proj/down_proj with all-reduce.
"""
from __future__ import annotations

import math
from dataclasses import dataclass, field
from typing import Optional

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.nn.modules.module import _has_any_global_hook

from helix_amd import ops
from helix_amd.models.meta import (DecodeMeta, KVLayer,  # noqa: F401
                                   MixedMeta, PrefillMeta)
from helix_amd.models.quant import FP8Linear
from helix_amd.ops import make_cos_sin_cache


@dataclass
class LlamaConfig:
    name: str = "llama3-8b"
    vocab_size: int = 128256
    hidden_size: int = 4096
    intermediate_size: int = 14336
    num_layers: int = 32
    num_heads: int = 32
    num_kv_heads: int = 8
    head_dim: int = 128
    rms_norm_eps: float = 1e-5
    rope_base: float = 500000.0
    max_position: int = 8192
    tie_embeddings: bool = False
    sliding_window: int = 0        # 0 = full attention (Mistral v0.1: 4096)
    attention_bias: bool = False   # Qwen2-style QKV bias
    rope_scaling: dict = field(default_factory=dict)  # llama3.1 scheme

    @property
    def q_size(self) -> int:
        return self.num_heads * self.head_dim

    @property
    def kv_size(self) -> int:
        return self.num_kv_heads * self.head_dim

    def kv_layers(self, tp_size: int = 1) -> list:
        return [KVLayer(self.num_kv_heads // tp_size, self.head_dim,
                        self.head_dim)] * self.num_layers

    def num_weights(self) -> tuple:
        """(embedding and head, per-layer total) parameter counts."""
        emb = self.vocab_size * self.hidden_size * \
            (1 if self.tie_embeddings else 2)
        per_layer = (self.hidden_size * (self.q_size + 2 * self.kv_size)
                     + self.q_size * self.hidden_size
                     + 3 * self.hidden_size * self.intermediate_size)
        return emb, self.num_layers * per_layer

    def activation_bytes(self, tokens: int) -> int:
        return 0            # covered by the memory-utilization margin

    @classmethod
    def from_json(cls, d: dict, name: str = "llama") -> "LlamaConfig":
        """From a Hugging Face config.json (llama, mistral, qwen2)."""
        heads = d["num_attention_heads"]
        qwen = (d.get("architectures") or [""])[0].startswith("Qwen2")
        window = d.get("sliding_window") or 0
        if not d.get("use_sliding_window", not qwen):
            window = 0
        return cls(
            name=name, vocab_size=d["vocab_size"],
            hidden_size=d["hidden_size"],
            intermediate_size=d["intermediate_size"],
            num_layers=d["num_hidden_layers"], num_heads=heads,
            num_kv_heads=d.get("num_key_value_heads") or heads,
            head_dim=d.get("head_dim") or d["hidden_size"] // heads,
            rms_norm_eps=d.get("rms_norm_eps", 1e-5),
            rope_base=float(d.get("rope_theta", 10000.0)),
            max_position=d.get("max_position_embeddings", 8192),
            tie_embeddings=d.get("tie_word_embeddings", False),
            sliding_window=window,
            attention_bias=d.get("attention_bias", qwen),
            rope_scaling=d.get("rope_scaling") or {})


PRESETS = {
    "llama3-8b": LlamaConfig(),
    # Llama-3.1: same weights shape as 3.0 but 128k context via the
    # llama3 rope-scaling scheme (HF config.json rope_scaling)
    "llama3.1-8b": LlamaConfig(
        name="llama3.1-8b", max_position=32768, rope_base=500000.0,
        rope_scaling={"rope_type": "llama3", "factor": 8.0,
                      "low_freq_factor": 1.0, "high_freq_factor": 4.0,
                      "original_max_position_embeddings": 8192}),
    "llama3-70b": LlamaConfig(
        name="llama3-70b", hidden_size=8192, intermediate_size=28672,
        num_layers=80, num_heads=64, num_kv_heads=8),
    "mistral-7b": LlamaConfig(
        name="mistral-7b", vocab_size=32000, rope_base=10000.0,
        sliding_window=4096),
    # Tiny configs for CPU tests and smoke runs.
    "tiny": LlamaConfig(
        name="tiny", vocab_size=512, hidden_size=256, intermediate_size=512,
        num_layers=2, num_heads=4, num_kv_heads=2, head_dim=64,
        max_position=512, rope_base=10000.0),
    "tiny-gqa": LlamaConfig(
        name="tiny-gqa", vocab_size=1024, hidden_size=512,
        intermediate_size=1024, num_layers=4, num_heads=8, num_kv_heads=2,
        head_dim=64, max_position=1024, rope_base=10000.0),
    "qwen2-7b": LlamaConfig(
        name="qwen2-7b", vocab_size=152064, hidden_size=3584,
        intermediate_size=18944, num_layers=28, num_heads=28,
        num_kv_heads=4, head_dim=128, rope_base=1000000.0,
        max_position=32768, attention_bias=True),
    "tiny-qwen": LlamaConfig(
        name="tiny-qwen", vocab_size=512, hidden_size=256,
        intermediate_size=512, num_layers=2, num_heads=4, num_kv_heads=2,
        head_dim=64, max_position=512, rope_base=10000.0,
        attention_bias=True),
    "tiny-sw": LlamaConfig(
        name="tiny-sw", vocab_size=512, hidden_size=256,
        intermediate_size=512, num_layers=2, num_heads=4, num_kv_heads=2,
        head_dim=64, max_position=512, rope_base=10000.0,
        sliding_window=24),
}


_WRITTEN = {}                     # class -> its forward as written


def _written(kind: type) -> type:
    _WRITTEN[kind] = kind.forward
    return kind


_written(FP8Linear)


@_written
class HLinear(nn.Linear):
    """nn.Linear routed through ops.linear: owned MFMA kernels, for a few rows
    by streamed weights, else by tiles; sizes and calls they do not take, or not
    as fast, stay with torch's.

    A plain call returns rows [T, N]. The modules here ask each other for
    other forms (_own says when): "sums" -> what ops.linear_sums_or_rows
    gives, for a reader that adds it up; "glu" -> silu(first half) * second half."""

    def forward(self, x: torch.Tensor, form: str = "rows") -> torch.Tensor:
        if self.bias is None and form == "sums":
            return ops.linear_sums_or_rows(x, self.weight)
        if self.bias is None and form == "glu":
            return ops.gated_linear(x, self.weight)
        out = ops.linear(x, self.weight, self.bias)
        return ops.silu_and_mul(out) if form == "glu" else out


def _own(m: nn.Module, *kinds: type) -> bool:
    """Whether m is one of these modules as written here: a subclass, a module
    put in its place, a forward put in place of its class's or a hook gets and
    returns what torch's linear would, [T, N], and never a form."""
    kind = type(m)
    if kind not in kinds or \
            kind.forward is not _WRITTEN.get(kind, kind.forward):
        return False
    d = m.__dict__
    return not (d["_forward_hooks"] or d["_forward_pre_hooks"]
                or "forward" in d or _has_any_global_hook())


def _project(proj: nn.Module, x: torch.Tensor, form: str) -> torch.Tensor:
    """proj(x) in that form; other kinds of projections know only rows."""
    if _own(proj, HLinear, FP8Linear):
        return proj(x, form)
    out = proj(x)
    return ops.silu_and_mul(out) if form == "glu" else out


@_written
class Attention(nn.Module):
    def __init__(self, cfg: LlamaConfig, tp_size: int = 1, tp_rank: int = 0):
        super().__init__()
        self.cfg = cfg
        assert cfg.num_heads % tp_size == 0 and cfg.num_kv_heads % tp_size == 0
        self.nh = cfg.num_heads // tp_size
        self.nkv = cfg.num_kv_heads // tp_size
        self.hd = cfg.head_dim
        self.scale = self.hd ** -0.5
        self.tp_size = tp_size
        self.window = cfg.sliding_window or 0
        q, kv, h = self.nh * self.hd, self.nkv * self.hd, cfg.hidden_size
        self.qkv_proj = HLinear(h, q + 2 * kv, bias=cfg.attention_bias)
        self.o_proj = HLinear(q, h, bias=False)

    def forward(self, x: torch.Tensor, cos_sin: torch.Tensor, kv_cache,
                meta, form: str = "rows", join=None,
                rows=None) -> torch.Tensor:
        """join (residual, norm_w, eps): few rows, see DecoderLayer. rows: those
        of the result that are asked for (None: all)."""
        T = x.shape[0]
        # fused strided split + rope + paged-cache write (one kernel, no
        # .contiguous() copies); compact K/V emitted only when the
        # fresh-prefill attention path consumes them directly
        mixed = isinstance(meta, MixedMeta)
        prefill = meta.prefill if mixed else meta
        want_kv = meta.is_prefill and \
            getattr(prefill, "cu_seqlens_k", None) is None
        heads = (cos_sin, self.nh, self.nkv, self.hd, kv_cache,
                 meta.slot_mapping, want_kv)
        if join is not None:
            q, k, v = ops.rows_qkv(meta.positions, x, self.qkv_proj.weight,
                                   self.qkv_proj.bias, *heads)
        else:
            q, k, v = self._heads(x, meta.positions, heads)
        if mixed:
            n = meta.num_decode
            o = torch.empty_like(q)
            both = self._attends_as_here()
            if want_kv:
                k, v = k[n:], v[n:]
            elif both:
                k, v = self._gather(q, kv_cache, prefill)
            if not (both and self._attend_both(q, k, v, kv_cache, meta, o)):
                self._attend_decode(q[:n], kv_cache, meta.decode, o[:n])
                self._attend_prefill(q[n:], k, v, kv_cache, prefill, o[n:])
        elif meta.is_prefill:
            o = self._attend_prefill(q, k, v, kv_cache, meta)
        else:
            o = self._attend_decode(q, kv_cache, meta)
        o = o.view(T, -1)
        if rows is not None:
            o = o[rows]
        if join is not None:
            return ops.rows_join(o, self.o_proj.weight, *join)
        if self.tp_size > 1:
            from helix_amd import parallel
            return parallel.tp_all_reduce(self.o_proj(o))
        return _project(self.o_proj, o, form)

    def _heads(self, x, positions, heads):
        """Turned and cached heads of x: of a few rows in the projection's launch."""
        p = self.qkv_proj
        if x.shape[0] <= ops.ROWS_QKV:
            if _own(p, HLinear) and \
                    ops.rows_qkv_fit(x, p.weight, p.bias, self.hd):
                return ops.rows_qkv(positions, x, p.weight, p.bias, *heads)
            if _own(p, FP8Linear) and isinstance(x, ops.Quantized) and \
                    ops.rows_qkv_fit(x, p.weight8, None, self.hd):
                return ops.rows_qkv(positions, x, p.weight8, None, *heads,
                                    w_scale=p.w_scale)
        return ops.rope_qkv_cache(positions, _project(p, x, "sums"), *heads)

    @staticmethod
    def _gather(q, kv_cache, meta):
        """Full-context K/V of a cached-prefix prefill, gathered from the paged
        cache (new tokens were just written)."""
        return ops.gather_kv(*kv_cache, meta.gather_blk, meta.gather_off,
                             q.dtype)

    def _attends_as_here(self) -> bool:
        """Whether nobody has put a way to attend of their own in place of these."""
        return all(name not in self.__dict__ and
                   getattr(type(self), name) is getattr(Attention, name)
                   for name in ("_attend_prefill", "_attend_decode"))

    def _attend_both(self, q, k, v, kv_cache, meta, out) -> bool:
        """Replies and portions in one launch, or False and nothing done."""
        n, d, p = meta.num_decode, meta.decode, meta.prefill
        if not (d.workspace and d.max_len):
            return False
        tmp_out, tmp_ml = d.workspace
        cu_k = p.cu_seqlens if p.cu_seqlens_k is None else p.cu_seqlens_k
        return ops.mixed_attention(
            (out[n:], q[n:], k, v, p.cu_seqlens, cu_k, p.max_seqlen),
            (out[:n], q[:n], *kv_cache, d.block_tables, d.seq_lens,
             tmp_out[:n], tmp_ml[:n], d.max_len), self.scale, self.window)

    def _attend_prefill(self, q, k, v, kv_cache, meta, out=None):
        """k and v of all tokens; None: to be gathered."""
        if k is None:
            k, v = self._gather(q, kv_cache, meta)
        return ops.attn_prefill(q, k, v, meta.cu_seqlens,
                                meta.max_seqlen, self.scale,
                                window=self.window,
                                cu_seqlens_k=meta.cu_seqlens_k, out=out)

    def _attend_decode(self, q, kv_cache, meta, out=None):
        k_cache, v_cache = kv_cache
        return ops.paged_attn_decode(q, k_cache, v_cache, meta.block_tables,
                                     meta.seq_lens, self.scale,
                                     meta.workspace, meta.max_len or None,
                                     window=self.window, out=out)


@_written
class MLP(nn.Module):
    def __init__(self, cfg: LlamaConfig, tp_size: int = 1):
        super().__init__()
        assert cfg.intermediate_size % tp_size == 0
        self.tp_size = tp_size
        i = cfg.intermediate_size // tp_size
        self.gate_up_proj = HLinear(cfg.hidden_size, 2 * i, bias=False)
        self.down_proj = HLinear(i, cfg.hidden_size, bias=False)

    def forward(self, x: torch.Tensor, form: str = "rows",
                join=None) -> torch.Tensor:
        """x Unscaled: few rows, see DecoderLayer; join as of Attention."""
        if isinstance(x, ops.Unscaled):
            h = ops.rows_glu(x, self.gate_up_proj.weight)
        else:
            h = _project(self.gate_up_proj, x, "glu")
        if join is not None:
            return ops.rows_join(h, self.down_proj.weight, *join)
        if self.tp_size > 1:
            from helix_amd import parallel
            return parallel.tp_all_reduce(self.down_proj(h))
        return _project(self.down_proj, h, form)


def _norm_for(m: nn.Module, kind: type, proj: str):
    """The norm before m: where m as written here hands the rows to an 8-bit
    projection, and to nothing else, it writes their bytes."""
    bytes_ = _own(m, kind) and _own(getattr(m, proj), FP8Linear)
    return ops.fused_add_rms_norm_fp8 if bytes_ else ops.fused_add_rms_norm


@_written
class DecoderLayer(nn.Module):
    def __init__(self, cfg: LlamaConfig, tp_size: int = 1, tp_rank: int = 0):
        super().__init__()
        self.input_norm_w = nn.Parameter(torch.ones(cfg.hidden_size))
        self.post_norm_w = nn.Parameter(torch.ones(cfg.hidden_size))
        self.attn = Attention(cfg, tp_size, tp_rank)
        self.mlp = MLP(cfg, tp_size)
        self.eps = cfg.rms_norm_eps

    def unseen(self) -> bool:
        """Whether all within it is as written here: nobody sees its rows but those
        who ask for the result. Asked of a layer that is _own itself: a module
        around one may hand on the question, but not its answer."""
        a, m = self.attn, self.mlp
        return (_own(a, Attention) and _own(m, MLP) and all(
            _own(p, HLinear, FP8Linear) for p in
            (a.qkv_proj, a.o_proj, m.gate_up_proj, m.down_proj)))

    def few(self, x) -> bool:
        """Whether these rows go through the layer in launches that take norm,
        rotation and residual along (layer_rows.hip): all of it is as written
        here, and whole on this GPU."""
        a, m = self.attn, self.mlp
        if not (_own(a, Attention) and _own(m, MLP)
                and a.tp_size == m.tp_size == 1):
            return False
        ps = (a.qkv_proj, a.o_proj, m.gate_up_proj, m.down_proj)
        return (all(_own(p, HLinear) for p in ps)
                and all(p.bias is None for p in ps[1:])
                and ops._bias_fits(ps[0].bias, ps[0].weight)
                and ops.layer_rows_fit(x, *(p.weight for p in ps), a.hd))

    def forward(self, x, residual, cos_sin, kv_cache, meta,
                form: str = "rows", few: bool = False, after=None, rows=None):
        """form "sums": the result's stretches, for the next norm. few: as few()
        says; after (few): weight and eps of that norm, which the result then is but
        for its division (ops.Unscaled). rows: those that are asked for, where attn
        is as written here; the others leave behind attention."""
        if residual is None:
            residual = x.clone()
            h = ops.rms_norm(x, self.input_norm_w, self.eps)
        elif isinstance(x, ops.Unscaled):
            h = x
        else:
            h, residual = _norm_for(self.attn, Attention, "qkv_proj")(
                x, residual, self.input_norm_w, self.eps)
        if few:
            h = self.attn(h, cos_sin, kv_cache, meta,
                          join=(residual, self.post_norm_w, self.eps))
            join = None if after is None else (residual, *after)
            return self.mlp(h, form, join), residual
        extra = {"form": "sums"} if _own(self.attn, Attention) else {}
        if rows is not None:
            extra["rows"] = rows
        h = self.attn(h, cos_sin, kv_cache, meta, **extra)
        if rows is not None:
            residual = residual[rows]
        h, residual = _norm_for(self.mlp, MLP, "gate_up_proj")(
            h, residual, self.post_norm_w, self.eps)
        h = self.mlp(h, *([form] if _own(self.mlp, MLP) else []))
        return h, residual


@_written
class LlamaForCausalLM(nn.Module):
    paged_prefill = False        # cached prefixes are gathered
    extension = "_C"             # native library of its kernels

    def __init__(self, cfg: LlamaConfig, tp_size: int = 1, tp_rank: int = 0):
        super().__init__()
        self.cfg = cfg
        self.tp_size = tp_size
        self.tp_rank = tp_rank
        self.embed_tokens = nn.Embedding(cfg.vocab_size, cfg.hidden_size)
        self.layers = nn.ModuleList(
            [DecoderLayer(cfg, tp_size, tp_rank) for _ in range(cfg.num_layers)])
        self.final_norm_w = nn.Parameter(torch.ones(cfg.hidden_size))
        if cfg.tie_embeddings:
            self.lm_head = None
        else:
            self.lm_head = HLinear(cfg.hidden_size, cfg.vocab_size,
                                   bias=False)
        cs = make_cos_sin_cache(cfg.head_dim, cfg.max_position, cfg.rope_base,
                                rope_scaling=cfg.rope_scaling or None)
        self.register_buffer("cos_sin", cs, persistent=False)

    def _apply(self, fn, recurse=True):
        # keep the RoPE table fp32 through .to(bfloat16) casts — the HIP
        # kernel consumes fp32 cos/sin.
        super()._apply(fn, recurse)
        if self.cos_sin.dtype != torch.float32:
            self.cos_sin = self.cos_sin.float()
        return self

    @torch.inference_mode()
    def forward(self, input_ids: torch.Tensor, kv_caches, meta) -> torch.Tensor:
        return self._hidden(input_ids, kv_caches, meta)

    @torch.inference_mode()
    def forward_rows(self, input_ids: torch.Tensor, kv_caches, meta,
                     rows: torch.Tensor) -> torch.Tensor:
        """Rows of what forward returns. Of a prompt, scores of the last token are
        asked for: the others end with the last layer's attention, whose
        feed-forward is 2 to 3% of all products. To take rows apart costs two
        launches, so this is for prompts of which at least half leave."""
        if input_ids.shape[0] >= 256 and \
                0 < 2 * rows.numel() <= input_ids.shape[0] and \
                _own(self, LlamaForCausalLM) and \
                _own(self.layers[-1], DecoderLayer) and \
                self.layers[-1].unseen():
            return self._hidden(input_ids, kv_caches, meta, rows)
        return self(input_ids, kv_caches, meta)[rows]

    def _few(self, i: int, x) -> bool:
        """Whether layer i takes rows as x are, of the first layer, in launches of a
        few; None: they are more."""
        if x is None or i >= len(self.layers):
            return False
        layer = self.layers[i]
        return _own(layer, DecoderLayer) and layer.few(x)

    def _hidden(self, input_ids, kv_caches, meta, rows=None) -> torch.Tensor:
        x = self.embed_tokens(input_ids)
        residual, own = None, True
        # asked a layer ahead and not of all at once, which is 12 us of the host
        # a layer (32 layers, eager, 14 tokens 4.24 ms and 3.84)
        first = x if x.shape[0] <= ops.LAYER_ROWS else None
        after = self._few(0, first)
        for i, layer in enumerate(self.layers):
            cache = kv_caches[i] if kv_caches is not None else None
            own = _own(layer, DecoderLayer)
            extra = {"form": "sums"} if own else {}
            few, after = after, self._few(i + 1, first)
            if few:
                then = self.layers[i + 1] if after else None
                extra.update(few=True, after=then and (then.input_norm_w,
                                                       then.eps))
            elif rows is not None and i + 1 == len(self.layers):
                extra["rows"] = rows
            x, residual = layer(x, residual, self.cos_sin, cache, meta, **extra)
        if not own:                # what a hook has kept stays as it was
            x, residual = x.clone(), residual.clone()
        return ops.fused_add_rms_norm(x, residual, self.final_norm_w,
                                      self.cfg.rms_norm_eps)[0]

    @torch.inference_mode()
    def compute_logits(self, hidden: torch.Tensor) -> torch.Tensor:
        if self.lm_head is not None:
            return self.lm_head(hidden)
        return F.linear(hidden, self.embed_tokens.weight)

    def decode_workspace(self, max_batch: int, max_len: int, device):
        return ops.decode_workspace(max_batch,
                                    self.cfg.num_heads // self.tp_size,
                                    self.cfg.head_dim, max_len, device)

    @torch.inference_mode()
    def init_random(self, seed: int = 0):
        """Random-init weights (no network => no real checkpoints).

        CPU path is generator-deterministic (tests build identical twins);
        GPU path inits in-place at device speed (8B+ scale).
        """
        std = 0.02
        on_gpu = next(self.parameters()).is_cuda
        if on_gpu:
            torch.cuda.manual_seed(seed)
        g = None if on_gpu else torch.Generator().manual_seed(seed)
        for name, p in self.named_parameters():
            if name.endswith("norm_w"):
                p.data.fill_(1.0)
            elif name.endswith(".bias"):
                p.data.zero_() if on_gpu else p.data.copy_(
                    torch.zeros(p.shape, dtype=torch.float32).to(p.dtype))
            elif on_gpu:
                p.data.normal_(0.0, std)
            else:
                t = torch.empty(p.shape, dtype=torch.float32)
                t.normal_(0.0, std, generator=g)
                p.data.copy_(t.to(p.dtype))
        return self

    def memory_bytes(self) -> int:
        return sum(p.numel() * p.element_size() for p in self.parameters())
