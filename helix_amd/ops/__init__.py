"""helix_amd.ops — CDNA4 (gfx950) kernel dispatch.

GPU tensors run the hand-written HIP kernels in helix_amd._C and FAIL
LOUDLY if the extension is missing (no silent eager fallback on a GPU
box). CPU tensors use the pure-torch reference implementations so engine
logic is testable without a GPU.
"""
from __future__ import annotations

import functools
import os
from typing import NamedTuple
from dataclasses import dataclass

import torch

from . import build
from . import reference as ref
from .reference import (banded_frequencies, make_cos_sin_cache,  # re-export
                        yarn_frequencies)

_C = None
_C_ERR: str | None = None
try:
    from helix_amd import _C  # type: ignore  # noqa: F401
    from helix_amd import _C as _C_mod
    _C = _C_mod
except ImportError as e:  # pragma: no cover
    _C_ERR = str(e)

def _native():
    if _C is None:
        raise RuntimeError(
            "helix_amd._C native extension is not built but a GPU tensor was "
            "passed. Build it with `python setup.py build_ext --inplace` "
            f"(PYTORCH_ROCM_ARCH=gfx950). Import error: {_C_ERR}")
    return _C


def _native_ext():
    return build.load("_C_ext")


def have_native(name: str = "_C") -> bool:
    if name == "_C":
        return _C is not None
    try:
        return build.load(name) is not None
    except RuntimeError:
        return False


def rms_norm(x: torch.Tensor, w: torch.Tensor, eps: float) -> torch.Tensor:
    if x.is_cuda:
        out = torch.empty_like(x)
        _native().rms_norm(out, x, w, eps)
        return out
    return ref.rms_norm(x, w, eps)


def fused_add_rms_norm(x: torch.Tensor, residual: torch.Tensor,
                       w: torch.Tensor, eps: float):
    """In-place on GPU: x <- norm(x+res), residual <- x+res. Returns both.
    On GPU x may be the stretches of a product (linear_sums, fp32
    [n, T, H]), which stay as they are."""
    if x.is_cuda and x.dim() == 3 and x.dtype == torch.float32:
        h = torch.empty_like(residual)
        _native().add_sums_rms_norm(h, x, residual, w, eps)
        return h, residual
    if x.is_cuda:
        _native().fused_add_rms_norm(x, residual, w, eps)
        return x, residual
    out, new_res = ref.fused_add_rms_norm(x, residual, w, eps)
    x.copy_(out)
    residual.copy_(new_res)
    return x, residual


class Quantized(NamedTuple):
    """Rows as e4m3 bytes and a float32 scale of each (quantize_fp8)."""
    bytes: torch.Tensor
    scales: torch.Tensor

    @property
    def shape(self):
        return self.bytes.shape


def fused_add_rms_norm_fp8(x: torch.Tensor, residual: torch.Tensor,
                           w: torch.Tensor, eps: float):
    """fused_add_rms_norm for 8-bit projections alone: stretches on GPU give
    Quantized rows, what quantize_fp8 makes of the norm, in the same launch.
    Other forms of x as there."""
    if x.is_cuda and x.dim() == 3 and x.dtype == torch.float32:
        h = Quantized(torch.empty_like(residual, dtype=torch.uint8),
                      torch.empty(residual.shape[0], dtype=torch.float32,
                                  device=x.device))
        _native().add_sums_rms_norm_fp8(*h, x, residual, w, eps)
        return h, residual
    return fused_add_rms_norm(x, residual, w, eps)


def layer_norm(x: torch.Tensor, w: torch.Tensor, b: torch.Tensor,
               eps: float) -> torch.Tensor:
    if x.is_cuda:
        out = torch.empty_like(x)
        _native().layer_norm(out, x, w, b, eps)
        return out
    return ref.layer_norm(x, w, b, eps)


def add_layer_norm(x: torch.Tensor, y: torch.Tensor, w: torch.Tensor,
                   b: torch.Tensor, eps: float) -> torch.Tensor:
    """Layer norm of x + y."""
    if x.is_cuda:
        out = torch.empty_like(x)
        if _native().add_norm(None, out, x, y, None, w, b, 0, eps):
            return out
    return layer_norm((x.float() + y.float()).to(x.dtype), w, b, eps)


def modulated_norm(x: torch.Tensor, scale: torch.Tensor, shift: torch.Tensor,
                   L: int, eps: float, y: torch.Tensor | None = None,
                   gate: torch.Tensor | None = None,
                   y_bias: torch.Tensor | None = None):
    """(s, norm(s) (1 + scale) + shift), s = x + gate y (x without y). norm
    is a layer norm without weights; gate, scale and shift have a row for
    every L rows of x. y_bias: y is in stretches [n, T, H] (fp32) of a product
    that this bias belongs to."""
    if x.is_cuda:
        out = torch.empty_like(x)
        s = x if y is None else torch.empty_like(x)
        if _native().add_norm(None if y is None else s, out, x, y, gate,
                              scale, shift, L, eps, y_bias):
            return s, out
    if y_bias is not None:
        y = (y.sum(0) + y_bias.float()).to(x.dtype)
    if y is not None:
        x = gated_add(x, y, gate, L)
    h = x.shape[-1]
    n = layer_norm(x, torch.ones(h, dtype=x.dtype, device=x.device),
                   torch.zeros(h, dtype=x.dtype, device=x.device), eps)
    c, s = (t.repeat_interleave(L, dim=0) for t in (scale, shift))
    return x, (n * (1 + c) + s).to(x.dtype)


def gated_add(x: torch.Tensor, y: torch.Tensor, gate: torch.Tensor,
              L: int) -> torch.Tensor:
    """x + gate y; gate has a row for every L rows of x."""
    if x.is_cuda:
        out = torch.empty_like(x)
        if _native().gated_add(out, x, y, gate, L):
            return out
    g = gate.repeat_interleave(L, dim=0)
    return (x.float() + g.float() * y.float()).to(x.dtype)


def text_embed(ids: torch.Tensor, cu: torch.Tensor, word: torch.Tensor,
               pos: torch.Tensor, w: torch.Tensor, b: torch.Tensor, eps: float):
    """Layer norm of word[ids] + pos[place within the text], NaN where either is
    outside its table, or None for other forms than the kernel reads (the CPU's
    among them)."""
    if ids.is_cuda and word.dim() == 2:
        out = torch.empty(ids.shape[0], word.shape[1], dtype=torch.bfloat16,
                          device=ids.device)
        if _native().text_embed(out, ids, cu, word, pos, w, b, eps):
            return out
    return None


def text_pool(x: torch.Tensor, cu: torch.Tensor):
    """Rows cu[:-1] of x (fp32), each divided by its length, or None as above."""
    if x.is_cuda:
        out = torch.empty(cu.shape[0] - 1, x.shape[1], device=x.device,
                          dtype=torch.float32)
        if _native().text_pool(out, x, cu):
            return out
    return None


def text_block(x: torch.Tensor, cu: torch.Tensor, max_len: int, heads: int,
               scale: float, eps: float, params: list):
    """A block of the text encoder by one call (blocks.hip): attention and
    feed-forward, each with the norm of its sum, or None as above."""
    if x.is_cuda and not _seen_by_torch():
        return _native().text_block(x, cu, max_len, heads, scale, eps, params)
    return None


def text_block_first(x: torch.Tensor, cu: torch.Tensor, max_len: int,
                     heads: int, scale: float, eps: float, params: list):
    """text_block for one who only asks for the first row of each text: (those
    rows, cu of texts of a row each), or None as above. A text without tokens is
    NaN."""
    if x.is_cuda and not _seen_by_torch():
        out = _native().text_block_first(x, cu, max_len, heads, scale, eps,
                                         params)
        return tuple(out) or None
    return None


def image_block(x: torch.Tensor, y, gate, y_bias, mod: torch.Tensor,
                cu: torch.Tensor, L: int, heads: int, scale: float, eps: float,
                params: list, stretches: bool = False):
    """A block of the image model by one call (blocks.hip), (x, y, gate, y_bias)
    of a sum that is still to be taken, or None as above. stretches: y may be such
    as modulated_norm adds up, with a bias; else y_bias is None."""
    if x.is_cuda and not _seen_by_torch():
        out = _native().image_block(x, y, gate, y_bias, mod, cu, L, heads,
                                    scale, eps, params, stretches)
        if out:
            return (*out, None)[:4]
    return None


def _seen_by_torch() -> bool:
    """Whether something wants to see the steps one by one."""
    return (torch.jit.is_tracing() or torch.compiler.is_compiling()
            or torch.is_autocast_enabled("cuda"))


def image_rows(lat: torch.Tensor, patch: int, columns: int):
    """Patches of the latents [B, C, S, S] as rows of so many columns (bf16, zeros
    behind a patch), or None as above."""
    if lat.is_cuda and lat.dim() == 4:
        n = (lat.shape[2] // patch) * (lat.shape[3] // patch)
        out = torch.empty(lat.shape[0] * n, columns, dtype=torch.bfloat16,
                          device=lat.device)
        if _native().image_rows(out, lat, patch):
            return out
    return None


def image_velocity(rows: torch.Tensor, shape, patch: int, text: int):
    """Rows of the image tokens, behind so many of text in each image, as latents
    of that shape (fp32), or None as above."""
    if rows.is_cuda:
        out = torch.empty(shape, dtype=torch.float32, device=rows.device)
        if _native().image_velocity(out, rows, patch, text):
            return out
    return None


def image_tokens(ids: torch.Tensor, word: torch.Tensor, pos: torch.Tensor,
                 image: torch.Tensor, cond: torch.Tensor):
    """(x, cu): word[ids] and the image's rows, each with its place, image after
    image, and their boundaries; the mean of word[ids] is added to cond. None as
    above."""
    if ids.is_cuda and pos.dim() == 2:
        B, (L, h) = ids.shape[0], pos.shape
        x = torch.empty(B * L, h, dtype=torch.bfloat16, device=ids.device)
        cu = torch.empty(B + 1, dtype=torch.int32, device=ids.device)
        if _native().image_tokens(x, cond, cu, ids, word, pos, image):
            return x, cu
    return None


def time_embed(t: torch.Tensor, dim: int):
    """Sinusoidal embedding of times (bf16), or None as above."""
    if t.is_cuda and t.dim() == 1:
        out = torch.empty(t.shape[0], dim, dtype=torch.bfloat16,
                          device=t.device)
        if _native().time_embed(out, t):
            return out
    return None


def rotary_embedding(positions: torch.Tensor, q: torch.Tensor,
                     k: torch.Tensor, cos_sin: torch.Tensor, head_dim: int):
    """In-place on GPU. Returns (q, k)."""
    if q.is_cuda:
        _native().rotary_embedding(positions, q, k, cos_sin, head_dim)
        return q, k
    qo, ko = ref.rotary_embedding(positions, q, k, cos_sin, head_dim)
    q.copy_(qo)
    k.copy_(ko)
    return q, k


def kv_fp8_quant(t: torch.Tensor) -> torch.Tensor:
    """bf16 -> OCP e4m3 bytes (uint8 view), any shape."""
    return t.to(torch.float8_e4m3fn).view(torch.uint8)


def kv_fp8_dequant(t: torch.Tensor, dtype=torch.bfloat16) -> torch.Tensor:
    """OCP e4m3 bytes (uint8) -> dtype."""
    return t.view(torch.float8_e4m3fn).to(dtype)


def gather_kv(k_cache: torch.Tensor, v_cache: torch.Tensor,
              blk: torch.Tensor, off: torch.Tensor, dtype=torch.bfloat16):
    """Rows [T, Hkv, D] of a paged cache at offsets off of pages blk; e4m3
    bytes become dtype. Other places than int64 of the same GPU are for torch's
    indexing, as are caches of other types or packing."""
    if (k_cache.is_cuda and dtype == torch.bfloat16 and
            k_cache.dtype in (torch.bfloat16, torch.uint8) and
            k_cache.shape[3] % 8 == 0 and
            v_cache.dtype == k_cache.dtype and
            v_cache.shape == k_cache.shape and
            k_cache.is_contiguous() and v_cache.is_contiguous() and
            blk.shape == off.shape and blk.dim() == 1 and
            all(t.dtype == torch.int64 and t.is_contiguous() and
                t.device == k_cache.device for t in (blk, off)) and
            v_cache.device == k_cache.device and _aligned(k_cache, v_cache) and
            k_cache.get_device() == torch.cuda.current_device()):
        k = torch.empty(blk.numel(), k_cache.shape[1], k_cache.shape[3],
                        dtype=dtype, device=k_cache.device)
        v = torch.empty_like(k)
        _native().gather_kv(k, v, k_cache, v_cache, blk, off)
        return k, v
    k, v = k_cache[blk, :, off], v_cache[blk, :, off]
    if k.dtype == torch.uint8:
        k, v = kv_fp8_dequant(k, dtype), kv_fp8_dequant(v, dtype)
    return k, v


def rope_qkv_cache(positions: torch.Tensor, qkv: torch.Tensor,
                   cos_sin: torch.Tensor, num_q: int, num_kv: int,
                   head_dim: int, kv_cache=None, slot_mapping=None,
                   want_kv: bool = False):
    """Fused QKV epilogue: strided split + rope + paged-cache write. qkv is
    [T, C] or [T, heads, head_dim], or in fp32 the stretches [n, T, C] of that
    product (linear_sums).

    Returns (q [T, num_q, head_dim], k, v) — k/v are None unless
    want_kv (fresh-prefill path needs compact K/V for attn_prefill).
    """
    sums = qkv.dim() == 3 and qkv.dtype == torch.float32
    T = qkv.shape[1 if sums else 0]
    if qkv.is_cuda:
        dtype = torch.bfloat16
        q_out = torch.empty(T, num_q * head_dim, dtype=dtype,
                            device=qkv.device)
        k_out = v_out = None
        if want_kv:
            k_out = torch.empty(T, num_kv * head_dim, dtype=dtype,
                                device=qkv.device)
            v_out = torch.empty_like(k_out)
        kc = vc = None
        if kv_cache is not None:
            kc, vc = kv_cache
        _native().rope_qkv_cache(positions, qkv, q_out, kc, vc,
                                 slot_mapping, k_out, v_out, cos_sin,
                                 num_q, num_kv, head_dim)
        return (q_out.view(T, num_q, head_dim),
                k_out.view(T, num_kv, head_dim) if want_kv else None,
                v_out.view(T, num_kv, head_dim) if want_kv else None)
    # CPU reference composition (same semantics)
    q_sz, kv_sz = num_q * head_dim, num_kv * head_dim
    q, k, v = qkv.split([q_sz, kv_sz, kv_sz], dim=-1)
    q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
    q, k = rotary_embedding(positions, q, k, cos_sin, head_dim)
    q = q.view(T, num_q, head_dim)
    k = k.view(T, num_kv, head_dim)
    v = v.view(T, num_kv, head_dim)
    if kv_cache is not None:
        if kv_cache[0].dtype == torch.uint8:    # fp8 KV cache
            reshape_and_cache(kv_fp8_quant(k), kv_fp8_quant(v),
                              kv_cache[0], kv_cache[1], slot_mapping)
        else:
            reshape_and_cache(k, v, kv_cache[0], kv_cache[1], slot_mapping)
    return q, (k if want_kv else None), (v if want_kv else None)


def silu_and_mul(x: torch.Tensor) -> torch.Tensor:
    if x.is_cuda:
        i = x.shape[-1] // 2
        out = torch.empty(*x.shape[:-1], i, dtype=x.dtype, device=x.device)
        _native().silu_and_mul(out, x)
        return out
    return ref.silu_and_mul(x)


def gelu_tanh(x: torch.Tensor) -> torch.Tensor:
    if x.is_cuda:
        out = torch.empty_like(x)
        _native().gelu_tanh(out, x)
        return out
    return ref.gelu_tanh(x)


def reshape_and_cache(k: torch.Tensor, v: torch.Tensor,
                      k_cache: torch.Tensor, v_cache: torch.Tensor,
                      slot_mapping: torch.Tensor):
    if k.is_cuda:
        _native().reshape_and_cache(k, v, k_cache, v_cache, slot_mapping)
        return
    ref.reshape_and_cache(k, v, k_cache, v_cache, slot_mapping)


def attn_prefill(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                 cu_seqlens: torch.Tensor, max_seqlen: int,
                 scale: float, causal: bool = True,
                 window: int = 0,
                 cu_seqlens_k: torch.Tensor | None = None,
                 out: torch.Tensor | None = None) -> torch.Tensor:
    """Varlen attention. When cu_seqlens_k is given, q rows are the
    SUFFIX of each sequence (cached-prefix prefill): kv rows cover the
    full context and causal positions are offset by klen - qlen. out: a
    contiguous place for the result."""
    if cu_seqlens_k is None:
        cu_seqlens_k = cu_seqlens
    if q.is_cuda:
        if out is None:
            out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        _native().attn_prefill(out, q, k, v, cu_seqlens, cu_seqlens_k,
                               max_seqlen, scale, causal, window)
        return out
    o = ref.attn_prefill(q, k, v, cu_seqlens, max_seqlen, scale, causal,
                         window, cu_seqlens_k)
    return o if out is None else out.copy_(o)


# Tokens that decode attention cuts sequences in (must match UNIT in
# paged_rows.h).
DECODE_PARTITION = 128


def decode_workspace(max_batch: int, num_q_heads: int, head_dim: int,
                     max_seq_len: int, device) -> tuple[torch.Tensor, torch.Tensor]:
    """Persistent fp32 scratch for partitioned decode attention."""
    max_parts = max(1, (max_seq_len + DECODE_PARTITION - 1) // DECODE_PARTITION)
    tmp_out = torch.empty(max_batch, num_q_heads, max_parts, head_dim,
                          dtype=torch.float32, device=device)
    tmp_ml = torch.empty(max_batch, num_q_heads, max_parts, 2,
                         dtype=torch.float32, device=device)
    return tmp_out, tmp_ml


def paged_attn_decode(q: torch.Tensor, k_cache: torch.Tensor,
                      v_cache: torch.Tensor, block_tables: torch.Tensor,
                      seq_lens: torch.Tensor, scale: float,
                      workspace=None, max_len: int | None = None,
                      window: int = 0,
                      out: torch.Tensor | None = None) -> torch.Tensor:
    """out: a contiguous place for the result."""
    if q.is_cuda:
        if out is None:
            out = torch.empty_like(q)
        if max_len is None:
            max_len = int(seq_lens.max())   # host sync — pass max_len to avoid
        if workspace is None:
            workspace = decode_workspace(q.shape[0], q.shape[1], q.shape[2],
                                         max_len, q.device)
        tmp_out, tmp_ml = workspace
        _native().paged_attn_decode(out, q, k_cache, v_cache, block_tables,
                                    seq_lens, scale,
                                    tmp_out[:q.shape[0]], tmp_ml[:q.shape[0]],
                                    max_len, window)
        return out
    if k_cache.dtype == torch.uint8:            # fp8 KV cache
        k_cache = kv_fp8_dequant(k_cache)
        v_cache = kv_fp8_dequant(v_cache)
    o = ref.paged_attn_decode(q, k_cache, v_cache, block_tables, seq_lens,
                              scale, window)
    return o if out is None else out.copy_(o)


def mixed_attention(portions: tuple, replies: tuple, scale: float,
                    window: int) -> bool:
    """attn_prefill of portions (out, q, k, v, cu_seqlens, cu_seqlens_k,
    max_seqlen) and paged_attn_decode of replies (out, q, k_cache, v_cache,
    block_tables, seq_lens, tmp_out, tmp_ml, max_len) in one launch, or False
    and nothing done for what only those two take, or take faster."""
    if not portions[1].is_cuda:
        return False
    return _native().attn_mixed(*portions, *replies, scale, window)


def sample_tokens(logits: torch.Tensor, temperatures: torch.Tensor,
                  seeds: torch.Tensor) -> torch.Tensor:
    if logits.is_cuda:
        out = torch.empty(logits.shape[0], dtype=torch.int64,
                          device=logits.device)
        _native().sample_tokens(out, logits, temperatures, seeds)
        return out
    return ref.sample_tokens(logits, temperatures, seeds)


def sample_tokens_ext(logits: torch.Tensor, temperatures: torch.Tensor,
                      seeds: torch.Tensor, top_p: torch.Tensor,
                      top_k: torch.Tensor, rep_pen: torch.Tensor,
                      pres_pen: torch.Tensor, freq_pen: torch.Tensor,
                      counts=None, seen=None, row_map=None) -> torch.Tensor:
    """Fused top-k/top-p/penalty Gumbel sampling (GPU only): one block
    per row, histogram-located threshold, no vocab sort. Penalties read
    per-row token-count tables indexed by row_map (engine row slots)."""
    out = torch.empty(logits.shape[0], dtype=torch.int64,
                      device=logits.device)
    _native().sample_tokens_ext(out, logits, temperatures, seeds, top_p,
                                top_k, rep_pen, pres_pen, freq_pen,
                                counts, seen, row_map)
    return out


def quantize_fp8(t: torch.Tensor, dim: int = -1):
    """Per-row (dim=-1 reduces over the last axis) e4m3 quantization.
    Returns (bytes uint8 view, float32 scales)."""
    if t.is_cuda and t.dtype == torch.bfloat16 and t.dim() == 2 and \
            dim in (-1, 1) and t.shape[1] > 0 and t.shape[1] % 8 == 0 and \
            t.is_contiguous() and _aligned(t) and \
            t.get_device() == torch.cuda.current_device():
        q = torch.empty(t.shape, dtype=torch.uint8, device=t.device)
        scale = torch.empty(t.shape[0], dtype=torch.float32, device=t.device)
        _native().quantize_rows(q, scale, t)
        return q, scale
    amax = t.float().abs().amax(dim=dim, keepdim=True).clamp(min=1e-8)
    scale = amax / 448.0                      # e4m3fn max normal
    q = (t.float() / scale).to(torch.float8_e4m3fn)
    return q.view(torch.uint8), scale.squeeze(dim).float()


def gemm_fp8(x8: torch.Tensor, w8: torch.Tensor, x_scale: torch.Tensor,
             w_scale: torch.Tensor, bias: torch.Tensor | None = None,
             act: int = 0) -> torch.Tensor:
    """out[M,N] = dequant(x8 @ w8^T): e4m3 inputs as uint8 views with
    per-row activation scales and per-output-channel weight scales
    (epilogue dequant; MFMA runs at the 2x fp8 rate)."""
    M, N = x8.shape[0], w8.shape[0]
    if x8.is_cuda:
        out = torch.empty(M, N, dtype=torch.bfloat16, device=x8.device)
        if act == 0 and _rows_fit(x8, w8) and _bias_fits(bias, w8):
            _native().gemm_rows(out, x8, w8, bias, x_scale.contiguous(),
                                w_scale.contiguous())
            return out
        _native().gemm_fp8(out, x8, w8, x_scale.contiguous(),
                           w_scale.contiguous(), bias, act)
        return out
    xf = x8.view(torch.float8_e4m3fn).float() * x_scale[:, None]
    wf = w8.view(torch.float8_e4m3fn).float() * w_scale[:, None]
    out = xf @ wf.t()
    if bias is not None:
        out = out + bias.float()
    if act == 1:
        out = torch.nn.functional.gelu(out, approximate="tanh")
    return out.to(torch.bfloat16)


def gemm_bf16(x: torch.Tensor, w: torch.Tensor, bias=None,
              act: int = 0) -> torch.Tensor:
    """act(x @ w^T + bias), act 1: GELU (tanh). Up to 64 rows of a small deep
    matrix stream their weights instead of going by tiles (us with weights from
    memory, streamed and by tiles: 8 rows of 768 x 3072 7.9 and 8.9, of 1024 x
    4096 7.9 and 9.1; of 6144 x 1024 7.7 and 7.2, of 2048 x 8192 11.4 and 10.9,
    64 of 3072 x 768 7.9 and 6.4)."""
    if x.is_cuda:
        out = torch.empty(x.shape[0], w.shape[0], dtype=x.dtype,
                          device=x.device)
        if (w.dim() == 2 and w.shape[1] >= 2 * w.shape[0]
                and w.numel() <= 8 << 20 and _rows_fit(x, w, 64, grads=False)
                and x.dtype == torch.bfloat16 and _bias_fits(bias, w)):
            _native().gemm_rows(out, x, w, bias, None, None, act == 1)
        else:
            _native().gemm_bf16(out, x, w, bias, act)
        return out
    return ref.gemm_bf16(x, w, bias, act)


def gemm_bf16_many(x: torch.Tensor, ws: list, biases: list) -> list:
    """[x @ w^T + bias] for several matrices: up to 64 rows in one launch, which
    is bound by reading the matrices and not by starting (8 rows of 12 x 6144 x
    1024 and 2048 x 1024 91 us as 13 launches, 31 as one)."""
    if x.is_cuda and x.shape[0] <= 64:
        out = _native().gemm_rows_many(x, ws, biases)
        if out:
            return out
    return [gemm_bf16(x, w, b) for w, b in zip(ws, biases)]


# The earlier kernel for few rows: called directly, or by linear with
# HELIX_SKINNY_GEMM=1. Llama's projections ask linear_sums and linear_silu_mul
# first, so that switch compares little of a decode step.
_SKINNY_MAX_M = 1024
_SKINNY_SCRATCH: dict = {}        # device -> fp32 workspace tensor
_SKINNY_SWIZZLE = os.environ.get("HELIX_SKINNY_SWIZZLE", "1") == "1"
_SKINNY_ENABLED = os.environ.get("HELIX_SKINNY_GEMM", "0") == "1"


def _skinny_split(M: int, N: int, K: int) -> int:
    """Split-K factor: enough workgroups to put ~3 on each of the 256
    CUs (m97-structure occupancy), subject to K dividing into 64s."""
    bm = 128 if M > 64 else 64
    tiles = ((M + bm - 1) // bm) * ((N + 127) // 128)
    s = 1
    while s < 8 and tiles * s < 768 and K % (s * 2 * 64) == 0:
        s *= 2
    return s


def gemm_skinny_bf16(x: torch.Tensor, w: torch.Tensor, bias=None,
                     act: int = 0) -> torch.Tensor:
    """Decode-shape GEMM (M <= 1024): split-K skinny tiles, fused
    bias/act epilogue. Caller guarantees bf16 CUDA contiguous inputs."""
    M, K = x.shape
    N = w.shape[0]
    out = torch.empty(M, N, dtype=x.dtype, device=x.device)
    s = _skinny_split(M, N, K)
    scratch = None
    if s > 1:
        need = s * M * N
        key = x.device.index
        cur = _SKINNY_SCRATCH.get(key)
        if cur is None or cur.numel() < need:
            cur = torch.empty(need, dtype=torch.float32, device=x.device)
            _SKINNY_SCRATCH[key] = cur
        scratch = cur
    _native().gemm_skinny_bf16(out, x, w, bias, scratch, s, act,
                               1 if _SKINNY_SWIZZLE else 0)
    return out


ROWS_MAX_M = 128                  # of gemm_rows.hip
ROWS_ANY = 1 << 30                # of gemm_ring.h
ROWS_MAX_M_GLU = 64               # of its gated form
ROWS_CHUNK = 512                  # bytes


def _rows_fit(x: torch.Tensor, w: torch.Tensor, most: int = ROWS_MAX_M,
              grads: bool = True) -> bool:
    """Whether the kernel for a few rows takes x @ w^T, bf16 or e4m3 bytes.
    It knows nothing of gradients, so where it stands for torch's product
    (grads) bf16 only runs where there are none to be had."""
    if not x.is_cuda or x.dim() != 2 or x.shape[0] > most or w.dim() != 2 \
            or torch.jit.is_tracing():
        return False
    (M, K), (N, Kw) = x.shape, w.shape
    if M == 0 or N == 0 or N % 8 != 0 or not 0 < K == Kw:
        return False
    dtype = x.dtype
    if dtype == torch.bfloat16:
        if K * 2 % ROWS_CHUNK or grads and not torch.is_inference_mode_enabled():
            return False
    elif dtype != torch.uint8 or K % ROWS_CHUNK:
        return False
    return (dtype == w.dtype and x.is_contiguous() and w.is_contiguous()
            and x.get_device() == w.get_device() and _aligned(x, w)
            # those have to see torch's own
            and not torch.is_autocast_enabled("cuda")
            and not torch.compiler.is_compiling())


def _aligned(*ts: torch.Tensor) -> bool:
    """Whether these are memory, on 16-byte boundaries."""
    try:
        for t in ts:
            if t.data_ptr() & 15:
                return False
    except RuntimeError:           # within vmap and the like they have none
        return False
    return True


def _bias_fits(bias, w: torch.Tensor) -> bool:
    """Whether the kernel for a few rows reads this bias as it lies."""
    return bias is None or (
        bias.shape == w.shape[:1] and bias.dtype == torch.bfloat16
        and bias.device == w.device and bias.is_contiguous())


def linear(x: torch.Tensor, w: torch.Tensor, bias=None) -> torch.Tensor:
    """Projection dispatch: owned kernels in inference, everything else (CPU,
    gradients, other types and strides, odd dims) via torch/hipBLASLt.

    The lines are where both were measured equal, with weights from memory. Up
    to 16 rows stream their weights (28672 x 4096: 42 against 60 us), vocabularies
    and up to 48 rows of wide matrices where _streams_pay. From 17 rows on tiles
    (gemm_ring.h) take less than the library's product in most sizes: 64 rows of
    4096 x 14336 29 us and 39, 1540 of 4096 x 4096 48 and 52, 4100 of 4096 x
    14336 384 and 733. Where they do not, _tiles_pay sends the product back to
    what took less before. Up to 128 rows of most wide matrices, bound by their
    weights, are the library's (128 of 12288 x 4096: 33 and 32). The library's
    time jumps from size to size: beyond 192 rows tiles take up to a tenth more
    in some (300 of 6144 x 4096 31 and 29, 777 of 20480 x 5120 181 and 167) and
    a tenth to half less in the others."""
    if (_SKINNY_ENABLED and x.is_cuda and x.dtype == torch.bfloat16
            and x.dim() == 2
            and w.dtype == torch.bfloat16 and 0 < x.shape[0] <= _SKINNY_MAX_M
            and x.shape[1] % 64 == 0 and w.shape[0] % 16 == 0
            and x.is_contiguous() and w.is_contiguous()):
        return gemm_skinny_bf16(x, w, bias)
    if _rows_fit(x, w, ROWS_ANY) and _bias_fits(bias, w):
        M, (N, K) = x.shape[0], w.shape
        tiles = M > 16 and _ring_fits(N, K) and (
            _tiles_pay(M, N, K) or _tiles_apart_pay(M, N, K))
        if tiles or _streams_pay(M, N, K):
            out = torch.empty(M, N, dtype=x.dtype, device=x.device)
            if tiles:
                _native().gemm_bf16(out, x, w, bias, 0)
            else:
                _native().gemm_rows(out, x, w, bias, None, None)
            return out
    return torch.nn.functional.linear(x, w, bias)


def _streams_pay(M: int, N: int, K: int) -> bool:
    """Whether up to 64 rows that do not go by tiles stream their weights rather
    than take the library's product: up to 16 rows of up to 65536 columns, and
    deep narrow ones. Of rows 4 or 8 KB apart: workgroups that begin apart
    (gemm_rows.hip) read these from all channels at once, which the library's do
    not. us streamed and by the library: 16 rows of 128256 x 4096 175 and 186,
    of 65536 x 2048 48 and 66, 32 of 32000 x 4096 46 and 63, 48 of it 52 and 64, 32
    of 28672 x 4096 45 and 54 (64 of it 53 and 53, of 16384 x 4096 35 and 32; 16
    of 128256 x 8192 373 and 364, 32 of 62024 x 3584 88 and 79). From 33 rows on
    tiles of 4096 are faster still. Vocabularies, whose time by the library jumps
    from size to size: 1 row of 128256 x 768 38 and 45, of 151936 x 3584 194 and
    227, of 131072 x 3584 163 and 162 (16 of it 166 and 160, 1 of 131072 x 5120 232
    and 227); 24 of 100352 x 1024 44 and 136, 32 of 66048 x 3584 104 and 110; 64 of
    128256 x 2048 114 and 119."""
    if N > 65536 and 768 <= K <= 4096:
        return (M <= 8 or 16 < M <= 32
                or K in (2048, 4096) and M <= (64 if K == 2048 else 48))
    if K in (2048, 4096) and M > 16 and N >= 24576:
        return M <= 48
    return N <= 65536 if M <= 16 else M <= 64 and K >= 2 * N and N <= 8192


def _tiles_apart_pay(M: int, N: int, K: int) -> bool:
    """Whether 17 to 128 rows of a wide matrix go by tiles all the same: of rows a
    multiple of 8 KB apart, whose tiles begin apart (ring_turn in gemm_ring.h), and
    columns that fill the chip. us by tiles and by the library: 33 of 28672 x 4096
    41 and 53, 128 51 and 56, 61 of 128256 x 4096 183 and 209, 128 191 and 234, of
    57344 x 8192 164 and 184 (80 of 37888 x 4096 80 and 72, 33 of 28672 x 8192 110
    and 100; 64 of 20480 x 4096 47 and 41, of 12288 x 4096 26 and 25). Up to 32 rows
    where tiles of 128 columns leave at most 96 of 256 CUs idle in their last round,
    else streamed (24 of 28672 x 4096 40 and streamed 47, of 57344 x 4096 83 and
    94, of 128256 x 4096 182 and 186, but of 81920 x 4096 147 and 122, of 114688 x
    4096 206 and 166). Vocabularies of other rows likewise (32 of 128256 x 3584 156,
    streamed 174, library 180; 24 of 100352 x 3584 148, 142 and 172) but for those
    4 KB apart (128256 x 2048 115 and streamed 97), and from 33 rows on while the
    inner dimension is short (64 of 151936 x 1536 101, library 111; 48 of 131072 x
    2560 130 and 127, of 100352 x 3072 129 and 119)."""
    if not 16 < M <= ROWS_MAX_M:
        return False
    full = (N // -128) % 256 <= 96
    if N > 65536 and 768 <= K < 4096:
        return K != 2048 and full if M <= 32 else K <= 1536
    return (K % 4096 == 0 and N >= 24576
            and (M > 32 or K == 4096 and full))


def _tiles_pay(M: int, N: int, K: int) -> bool:
    """Whether more than 16 rows go by tiles of 64 x 64 and more rather than by
    the library's smaller ones or, up to 64 rows of a deep matrix, as streamed
    weights. us by tiles and by the other:
    - wide matrices are bound by their weights (128 of 12288 x 4096 33 and 32),
      see _tiles_apart_pay;
    - few columns, so that few CUs read the weights: 33 of 768 x 16384 14.6 and
      13.2 (streamed), of 1024 x 16384 15.3 and 14.4;
    - up to 128 tiles of a few dozen steps, which end before they have hidden
      their first loads: 64 of 2048 x 2048 10.1 and 9.4, 192 of 1024 x 2048 10.0
      and 8.9, 512 of 1024 x 1280 8.3 and 8.0 (577 of it 8.3 and 10.5; 128 of
      2560 x 2048 10.2 and 12.3, 24 of 1536 x 2048 7.6 and 8.7, 65 of 512 x 3072
      7.9 and 10.0);
    - the like of a dozen steps, 100 of 768 x 768 6.1 and 5.3, 32 of 1024 x 1024
      6.7 and 5.7 (193 of 768 x 768 6.1 and 7.2, 33 of 1280 x 1024 6.8 and 8.6);
    - rows 16 KB apart, which lie on the same channels: 32 of 8192 x 8192 38 and
      31, 100 of it 42 and 39, 24 of 7168 x 8192 35 and 28 (48 of it 34 and 33)."""
    if N > 8192:
        return M > ROWS_MAX_M
    if N <= 1024 and K >= 2048 and K >= 2 * N and M <= (
            64 if K >= 12288 else 48):
        return False
    tiles = -(-M // 64) * -(-N // 64)
    if 1024 < K <= 3072 and N * K <= 8 << 20 and tiles <= 128:
        return (K >= 2048 and tiles <= (16 if K > 2048 else 12)
                or N > 2048 and M % 128 == 0 or N <= 2048 <= K and M <= 24)
    if 512 < K <= 1024:
        return not (M <= 192 and N * K <= 11 << 16 and (N > 256 or K > 768)
                    or M <= 32 and N <= 1280)
    return not (K % 8192 == 0 and K < 2 * N and
                (M <= 32 and N >= 6144 or M < 128 and N == 8192))


def _ring_fits(N: int, K: int, gated: bool = False) -> bool:
    """Whether the offsets of gemm_ring.h reach a matrix [N, K]."""
    if gated:                     # both halves lie behind one descriptor
        return K <= 1 << 21 and N <= 1 << 21 and 2 * N * K < (1 << 31) - 1
    return K <= 1 << 21 and N <= 1 << 20


def linear_sums(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x @ w^T for a reader that adds up stretches of the inner dimension
    (fused_add_rms_norm, rope_qkv_cache): [stretches, M, N] fp32 for up to 128
    rows and up to 8192 columns, and for more rows where _sums_pay; else [M, N]
    in x's type. Wide matrices fill the chip without stretches, whose sums are
    more bytes than they save."""
    M = x.shape[0]
    if _rows_fit(x, w, SUMS_MAX_M) and w.shape[0] <= 8192:
        tiles = x.dtype == torch.bfloat16 and _ring_fits(*w.shape)
        if M <= ROWS_MAX_M and (not tiles or _sums_streamed(M, *w.shape)):
            return _native().gemm_rows_sums(x, w, None, None)
        if tiles and (M <= ROWS_MAX_M or _sums_pay(M, *w.shape)):
            return _native().gemm_bf16_sums(x, w, 0)
    return linear(x, w)


def linear_sums_or_rows(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """linear_sums where stretches are the faster form for its reader, rows
    [M, N] elsewhere."""
    if x.dim() == 2 and x.shape[0] > 64 and _rows_fit(x, w, ROWS_MAX_M) \
            and not _sums_pay(x.shape[0], *w.shape):
        return linear(x, w)
    return linear_sums(x, w)


SUMS_MAX_M = 2048


def _sums_streamed(M: int, N: int, K: int) -> bool:
    """Whether stretches of a few rows come from streamed weights rather than
    from tiles (us with the norm that reads them, streamed and by tiles): up to
    16 rows; small products, which tiles start later (33 of 1024 x 768 7.4 and
    8.2, 48 of 2048 x 2048 10.1 and 10.5; 17 of 3072 x 1536 10.2 and 9.8, 64 of
    1024 x 1024 8.9 and 8.5); deep ones of few columns (48 of 1024 x 16384 16.4
    and 17.7, of 1024 x 8192 12.3 and 11.4) and rows 16 KB apart (33 of 8192 x
    8192 38.4 and 42.6)."""
    if M <= 16:
        return True
    if N * K <= 4 << 20 and K <= 2560:
        return M <= (64 if K < 1024 else 48)
    if N <= 1024 and K >= 12288:
        return M <= 64
    return K % 8192 == 0 and K < 2 * N and (
        M <= 24 and N >= 7168 or M <= 64 and N == 8192)


@functools.lru_cache(maxsize=4096)
def _sums_pay(M: int, N: int, K: int) -> bool:
    """Whether more than 64 rows gain from stretches: by the estimates that
    choose their tiles (gemm_ring.h), with what a reader reads of either form. Half
    a microsecond is left to rows, and a fifth of them where they do not go by
    tiles. us with the norm that reads them, as rows and in stretches: 65 of 2048
    x 2048 11.8 and 10.4, 129 of 4096 x 4096 21.5 and 21.0, 200 of it 22.0 and
    20.7, 400 of it 28.2 and 30.3; 129 of 6144 x 4096 26.4 and 23.9; 200 of 4096
    x 14336 47 and 44, 1540 182 and 167. Over 3700 sizes of 65 to 8192 rows what
    it takes is 1.5% slower than the best form of each (100 of 512 x 1280, in
    stretches, 9.1 for the library's 7.6)."""
    if not _ring_fits(N, K):
        return M <= ROWS_MAX_M
    if M > SUMS_MAX_M or N > 8192:
        return False
    plan = _native().gemm_bf16_plan
    tile, stretches, rows, _ = plan(M, N, K, False, False)
    if stretches > 1:
        rows += 4                       # the launch that joins them
    if not _tiles_pay(M, N, K):
        rows *= 0.8
    return plan(M, N, K, False, True)[2] + 0.5 <= rows + 2 * M * N / 4.5e6


def _glu_fits(M: int, N: int, K: int) -> bool:
    """Whether the gated product of up to 64 rows takes no longer in one launch
    than product and activation apart: up to 16 rows by streamed weights, which
    are not cut along the inner dimension and so need columns enough to fill the
    chip, or few chunks; then by the same or by tiles (gated_linear). us apart and
    at once, with weights from memory: one row of 28672 x 4096 59 and 42, 10240 x
    4096 28 and 29, 4096 x 4096 18 and 27, 16384 x 1024 12.3 and 10.2. From 17 rows
    on x is read by every workgroup, and the product apart is the faster one but
    for rows of 4 or 8 KB, which the library's workgroups all read from the same
    channels at once: 64 of 28672 x 4096 56 and 46; 48 of 37888 x 3584 64 and 69,
    of 10240 x 8192 44 and 53. Widths that the activation alone does not take go
    here."""
    if K <= 1024 or N % 16 != 0:
        return True
    if M <= 16:
        return N >= 3 * K
    return N >= 13 << 11 and K in (2048, 4096)


def linear_silu_mul(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """silu(x @ gate^T) * (x @ up^T), w = [gate; up]. A few rows: one launch,
    whose halves stay in registers (42 us at one row of 2 x 14336 x 4096,
    product and activation apart 59)."""
    if _rows_fit(x, w, ROWS_MAX_M_GLU):
        out = torch.empty(x.shape[0], w.shape[0] // 2, dtype=x.dtype,
                          device=x.device)
        _native().gemm_rows_glu(out, x, w, None, None)
        return out
    return silu_and_mul(linear(x, w))


def gated_linear(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """linear_silu_mul where that is the faster form, product and activation
    apart elsewhere. From 33 rows on by tiles, whose halves meet before they are
    rounded: in one launch (us apart and now: 64 rows of 28672 x 4096 56 and 46,
    512 107 and 95, 8192 1407 and 1249), from 17 on where tiles of wide matrices
    begin apart (ring_turn in gemm_ring.h; us streamed and by tiles: 17 of 28672 x
    4096 43.8 and 43.6, 24 45.2 and 43.5, 32 46.9 and 43.8, of 26624 x 4096 46.4
    and 39.7, of 32768 x 4096 49.0 and 48.6, but 24 47.9 and 48.4), and where
    that leaves CUs idle, narrow or deep, in stretches that a second one adds up
    (apart, in one launch and now: 80 of 2048 x 8192 20, 43 and 15, 100 of 4096 x
    14336 43, 79 and 37, 512 of 1024 x 16384 50, 90 and 30). Up to 64 rows of more
    than 8192 columns, where _glu_fits does not take them, are bound by their
    weights and stay apart (48 of 10240 x 8192 53 in one launch, 44 apart; 64 of
    14336 x 4096 36 and 31)."""
    apart = 16 if w.dim() == 2 and w.shape[1] % 4096 == 0 and \
        w.shape[0] > 8192 else 32
    if x.dim() == 2 and w.dim() == 2 and x.shape[0] > apart and \
            w.shape[0] % 16 == 0 and x.dtype == torch.bfloat16 and (
                x.shape[0] > ROWS_MAX_M_GLU or w.shape[0] <= 8192 or
                _glu_fits(x.shape[0], *w.shape)) and \
            _ring_fits(*w.shape, gated=True) and _rows_fit(x, w, ROWS_ANY):
        out = torch.empty(x.shape[0], w.shape[0] // 2, dtype=x.dtype,
                          device=x.device)
        _native().gemm_bf16_glu(out, x, w)
        return out
    if x.dim() == 2 and w.dim() == 2 and not _glu_fits(x.shape[0], *w.shape):
        return silu_and_mul(linear(x, w))
    return linear_silu_mul(x, w)


class Unscaled(NamedTuple):
    """Rows times a norm's weight that are still to be divided by the root of
    their mean square, which is eps and the mean of squares' sum over a row: what
    multiplies them may do so last (layer_rows.hip)."""
    rows: torch.Tensor                  # [M, H] bf16
    squares: torch.Tensor               # [M, parts] fp32
    eps: float

    @property
    def shape(self):
        return self.rows.shape


LAYER_ROWS = 16                   # of layer_rows.hip


def layer_rows_fit(x, qkv: torch.Tensor, o: torch.Tensor,
                   gate_up: torch.Tensor, down: torch.Tensor,
                   head_dim: int) -> bool:
    """Whether a layer's four projections of these rows go by layer_rows.hip:
    sizes it takes, up to 4 rows of up to 8192 columns and up to 16 of up to
    4096. Beyond, its workgroups of 16 and 32 columns read x more often than the
    launches that they save are worth. us of the four with norms and rotation, apart
    and so: 1 row of 4096 (llama3-8b) 94.8 and 84.4, 16 101 and 96; of 3584
    (qwen2-7b) 115.6 and 100.9, 118 and 115; of 2048 with 2 x 8192 48.6 and 35.0,
    49.6 and 45.9; of 8192 (llama3-70b) 332 and 317, 8 334 and 336, 16 337 and 357;
    of 5120 with 2 x 13824 137 and 132, 8 142 and 144."""
    x = x.rows if isinstance(x, Unscaled) else x
    if not x.is_cuda or x.dim() != 2 or x.shape[0] > LAYER_ROWS:
        return False
    H = x.shape[1]
    return (H % 64 == 0 and H <= (4096 if x.shape[0] > 4 else 8192)
            and head_dim % 32 == 0
            and x.dtype == torch.bfloat16
            and o.dim() == 2 and down.dim() == 2
            and o.shape[0] == H and down.shape[0] == H
            and _rows_fit(x, qkv, LAYER_ROWS)
            and _rows_fit(x, gate_up, LAYER_ROWS)
            and gate_up.shape[0] % 64 == 0
            and gate_up.shape[0] == 2 * down.shape[1]
            and all(w.dtype == torch.bfloat16 and w.is_contiguous()
                    and w.shape[1] * 2 % ROWS_CHUNK == 0
                    and w.device == x.device and _aligned(w)
                    for w in (o, down)))


def rows_join(x: torch.Tensor, w: torch.Tensor, residual: torch.Tensor,
              norm_w: torch.Tensor, eps: float) -> Unscaled:
    """residual += x @ w^T; its norm times norm_w, but for the division."""
    return Unscaled(*_native().layer_rows_join(x, w, residual, norm_w), eps)


def rows_glu(x: Unscaled, w: torch.Tensor) -> torch.Tensor:
    """silu(first half) * second half of x's norm @ w^T."""
    return _native().layer_rows_glu(x.rows, w, x.squares, x.eps)


def rows_qkv(positions: torch.Tensor, x, w: torch.Tensor, bias,
             cos_sin: torch.Tensor, num_q: int, num_kv: int, head_dim: int,
             kv_cache=None, slot_mapping=None, want_kv: bool = False,
             w_scale: torch.Tensor | None = None):
    """rope_qkv_cache of x @ w^T + bias in one launch; x are rows or Unscaled, or
    Quantized where w are e4m3 bytes with a scale of each row."""
    squares, eps, x_scale = None, 0.0, None
    if isinstance(x, Unscaled):
        x, squares, eps = x
    elif isinstance(x, Quantized):
        x, x_scale = x
    T = x.shape[0]
    q = torch.empty(T, num_q, head_dim, dtype=torch.bfloat16, device=x.device)
    k = v = None
    if want_kv:
        k = torch.empty(T, num_kv, head_dim, dtype=q.dtype, device=x.device)
        v = torch.empty_like(k)
    kc, vc = kv_cache if kv_cache is not None else (None, None)
    _native().layer_rows_qkv(x, w, bias, squares, eps, positions, cos_sin, q, k,
                             v, kc, vc, slot_mapping, num_q, num_kv, head_dim,
                             x_scale, w_scale)
    return q, k, v


ROWS_QKV = 32                     # of layer_rows.hip, without squares


def rows_qkv_fit(x, w: torch.Tensor, bias, head_dim: int) -> bool:
    """Whether rows_qkv takes rows or Quantized ones, and takes no longer than the
    product in stretches with rope_qkv_cache: its workgroups read x more often, the
    more the more rows and the deeper they are, and tiles take over wide matrices
    from 17 rows on. us apart and at once: 1 row of 6144 x 4096 14.5 and 12.0, 32
    16.4 and 15.6; 16 of 15360 x 5120 37.8 and 36.2, 32 33.7 and 42; 4 of 10240 x
    8192 39.9 and 39.0, 8 39 and 47; 32 of 12288 x 4096 25 and 29. e4m3: 32 of 6144 x
    4096 13.4 and 10.3, of 15360 x 5120 25.8 and 23.9, 8 of 10240 x 8192 24.3 and
    23.9, 16 24.0 and 25.2."""
    bytes_ = isinstance(x, Quantized)
    x = x.bytes if bytes_ else x
    if not (_rows_fit(x, w, ROWS_QKV) and _bias_fits(bias, w)
            and head_dim % 32 == 0):
        return False
    (M, K), N = x.shape, w.shape[0]
    if bytes_:
        return K <= (8192 if M <= 8 else 5120)
    if M > 16:
        return K <= 4096 and N <= 8192
    return K <= (8192 if M <= 4 else 5120)


def gemm_fp8_sums(x8: torch.Tensor, w8: torch.Tensor, x_scale: torch.Tensor,
                  w_scale: torch.Tensor) -> torch.Tensor:
    """gemm_fp8 for a reader that adds up stretches (linear_sums)."""
    if _rows_fit(x8, w8) and w8.shape[0] <= 8192:
        return _native().gemm_rows_sums(x8, w8, x_scale, w_scale)
    return gemm_fp8(x8, w8, x_scale, w_scale)


def gemm_fp8_silu_mul(x8: torch.Tensor, w8: torch.Tensor,
                      x_scale: torch.Tensor,
                      w_scale: torch.Tensor) -> torch.Tensor:
    """silu(first half) * second half of gemm_fp8's columns."""
    if _rows_fit(x8, w8, ROWS_MAX_M_GLU):
        out = torch.empty(x8.shape[0], w8.shape[0] // 2,
                          dtype=torch.bfloat16, device=x8.device)
        _native().gemm_rows_glu(out, x8, w8, x_scale, w_scale)
        return out
    return silu_and_mul(gemm_fp8(x8, w8, x_scale, w_scale))


def mfma_probe(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    d = torch.empty(16, 16, dtype=torch.float32, device=a.device)
    _native().mfma_probe(d, a, b)
    return d


# ---------------------------------------------------------------------------
# Depth-averaged fp32 residual stream, PolyNorm, talking-head attention
# ---------------------------------------------------------------------------

@dataclass
class TalkParams:
    """Constants of one talking-head attention layer. softcap / window 0,
    slopes / talk None switch the mechanism off."""
    scale: float
    softcap: float = 0.0
    window: int = 0
    slopes: torch.Tensor | None = None     # [H] fp32 distance bias per head
    talk: torch.Tensor | None = None       # [H, H] fp32 mixing matrix

    def max_keys(self, max_len: int) -> int:
        return min(max_len, self.window) if self.window else max_len


def embed_norm(ids: torch.Tensor, embed: torch.Tensor, w: torch.Tensor,
               eps: float, x: torch.Tensor) -> torch.Tensor:
    """x (fp32, written) <- embed[ids]; returns its RMS norm times w."""
    if embed.is_cuda:
        h = torch.empty(x.shape, dtype=embed.dtype, device=x.device)
        _native_ext().embed_norm(h, x, ids, embed, w, eps)
        return h
    return ref.embed_norm(ids, embed, w, eps, x)


def depth_norm(x: torch.Tensor, y: torch.Tensor, hist: torch.Tensor,
               n_prev: int, coef: torch.Tensor, w: torch.Tensor, eps: float,
               store_new: bool = True,
               x_out: torch.Tensor | None = None) -> torch.Tensor:
    """Layer result X = x + y, depth average over hist[:n_prev] and X, RMS
    norm. Appends X to hist (store_new), writes the average to x_out (which
    may be x), returns the normed rows in y's dtype."""
    if y.is_cuda:
        h = torch.empty(x.shape, dtype=y.dtype, device=y.device)
        _native_ext().depth_norm(h, x_out, x, y, hist, n_prev, store_new,
                                 coef, w, eps)
        return h
    return ref.depth_norm(x, y, hist, n_prev, coef, w, eps, store_new, x_out)


def poly_norm(z: torch.Tensor, coef: torch.Tensor, eps: float,
              out: torch.Tensor | None = None) -> torch.Tensor:
    """a N(z) + b N(z^2) + c N(z^3) + e, N = division by the row's root
    mean square; coef = (a, b, c, e) fp32. z and out may be column slices."""
    if out is None:
        out = torch.empty(z.shape, dtype=z.dtype, device=z.device)
    if z.is_cuda:
        _native_ext().poly_norm(out, z, coef, eps)
    else:
        out.copy_(ref.poly_norm(z, coef, eps))
    return out


def unit_qkv_cache(z: torch.Tensor, offsets, num_q: int, head_dim: int,
                   kv_cache, slot_mapping: torch.Tensor, eps: float,
                   v_first: torch.Tensor | None = None,
                   lam: torch.Tensor | None = None, first: bool = False,
                   ff=None) -> torch.Tensor:
    """Epilogue of the fused input projection z: unit-RMS q and k heads (no
    weight), value mixing, paged-cache write; returns q [T, H, Dp].

    offsets = (q, k, v) column starts. lam switches value mixing on: the
    first such layer writes its values to v_first, later ones blend
    (1 - lam) v + lam v_first. ff = (z_cols, out_cols, coef) runs PolyNorm
    in the same launch. Cache: K [nblk, G, bs, Dp], V [nblk, G, E, bs].
    """
    kc, vc = kv_cache
    if z.is_cuda:
        q = torch.empty(z.shape[0], num_q, kc.shape[3], dtype=z.dtype,
                        device=z.device)
        args = (z, *offsets, q, kc, vc, slot_mapping, v_first, lam, first,
                head_dim, eps)
        if ff is None:
            _native_ext().unit_qkv_cache(*args)
        else:
            zf, out, coef = ff
            _native_ext().layer_epilogue(*args, out, zf, coef)
        return q
    if ff is not None:
        zf, out, coef = ff
        out.copy_(ref.poly_norm(zf, coef, eps))
    return ref.unit_qkv_cache(z, offsets, num_q, head_dim, kc, vc,
                              slot_mapping, eps, v_first, lam, first)


# Partition granularity of the row kernels (QUANT in talk_attn_rows.hip) and
# their scratch bound when they process a whole prompt.
TALK_PARTITION = 128
TALK_SCRATCH_FLOATS = 64 << 20


def _talk_parts(rows: int, num_kv: int, max_keys: int) -> int:
    return min(-(-max_keys // TALK_PARTITION),
               max(1, 1024 // max(1, rows * num_kv)))


def talk_scratch_floats(rows: int, num_q: int, num_kv: int, v_dim: int,
                        max_keys: int) -> int:
    parts = _talk_parts(rows, num_kv, max_keys)
    return rows * num_q * (max_keys + parts * (2 + v_dim))


def talk_attn_rows(out: torch.Tensor, q: torch.Tensor, kv_cache,
                   block_tables: torch.Tensor, row_len: torch.Tensor,
                   max_len: int, p: TalkParams, gate=None, row_seq=None,
                   workspace: torch.Tensor | None = None) -> None:
    """out [R, H*E] <- attention of single query rows; row r reads the
    first row_len[r] cached tokens of block-table row row_seq[r] (r if
    None). gate: [R, H] logits, one sigmoid factor per head."""
    kc, vc = kv_cache
    if not q.is_cuda:
        ref.talk_attn_rows(out, q, kc, vc, block_tables, row_len, p, gate,
                           row_seq)
        return
    R, H = q.shape[:2]
    G, E = vc.shape[1:3]
    keys = p.max_keys(max_len)
    need = talk_scratch_floats(R, H, G, E, keys)
    if workspace is None or workspace.numel() < need:
        workspace = torch.empty(need, dtype=torch.float32, device=q.device)
    parts = _talk_parts(R, G, keys)
    a, b = R * H * keys, R * H * parts * 2
    _native_ext().talk_attn_rows(
        out, q, kc, vc, block_tables, row_seq, row_len, keys, p.scale,
        p.softcap, p.window, p.slopes, p.talk, gate,
        workspace[:a].view(R, H, keys),
        workspace[a:a + b].view(R, H, parts, 2),
        workspace[a + b:need].view(R, H, parts, E))


def talk_attn_prefill(out: torch.Tensor, q: torch.Tensor, kv_cache,
                      block_tables: torch.Tensor, cu_seqlens: torch.Tensor,
                      seq_lens: torch.Tensor, max_q: int, max_len: int,
                      row_seq: torch.Tensor, row_len: torch.Tensor,
                      p: TalkParams, gate=None) -> None:
    """Prompt portions: sequence b's rows cu_seqlens[b]..[b+1] are the last
    ones of its seq_lens[b] cached tokens. bf16 runs the MFMA kernel; fp32
    and oversized heads run the row kernels in slices of bounded scratch
    (row_seq / row_len map each row to its sequence and visible length)."""
    kc, vc = kv_cache
    if not q.is_cuda:
        ref.talk_attn_rows(out, q, kc, vc, block_tables, row_len, p, gate,
                           row_seq)
        return
    T, H, Dp = q.shape
    G, E = vc.shape[1:3]
    if q.dtype == torch.bfloat16 and \
            _native_ext().talk_prefill_fits(H, Dp, E):
        talk = p.talk if p.talk is not None else torch.eye(
            H, device=q.device)
        lse = torch.empty(T, H, dtype=torch.float32, device=q.device)
        _native_ext().talk_attn_prefill(
            out, q, kc, vc, block_tables, cu_seqlens, seq_lens, max_q,
            p.scale, p.softcap, p.window, p.slopes, talk, gate, lse)
        return
    keys = p.max_keys(max_len)
    step = max(1, TALK_SCRATCH_FLOATS // (H * (keys + 2 + E)))
    for r in range(0, T, step):
        s = slice(r, min(T, r + step))
        talk_attn_rows(out[s], q[s], kv_cache, block_tables, row_len[s],
                       max_len, p, None if gate is None else gate[s],
                       row_seq[s])
