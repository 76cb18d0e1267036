"""bge-class BERT encoder for embeddings (feeds the RAG vector store).

Replaces the reference's delegated embedding models (kodit ONNX text
model / `/v1/embeddings` proxying, SURVEY.md §2.8 "Embedding models").
All projection GEMMs run on the hand-written MFMA bf16 GEMM
(ops.gemm_bf16, gemm_bf16.hip) with fused bias + GELU on the MLP up
projection; attention is the non-causal mode of the varlen flash kernel.
"""
from __future__ import annotations

from dataclasses import dataclass

import torch
import torch.nn as nn

from helix_amd import ops
from helix_amd.models.llama import _own, _written


@dataclass
class BertConfig:
    name: str = "bge-base"
    vocab_size: int = 30528          # padded to /64 for the MFMA GEMM
    hidden_size: int = 768
    intermediate_size: int = 3072
    num_layers: int = 12
    num_heads: int = 12
    max_position: int = 512
    layer_norm_eps: float = 1e-12
    pooling: str = "cls"             # cls | mean


BERT_PRESETS = {
    "bge-base": BertConfig(),
    "bge-large": BertConfig(name="bge-large", hidden_size=1024,
                            intermediate_size=4096, num_layers=24,
                            num_heads=16),
    "tiny-bert": BertConfig(name="tiny-bert", vocab_size=512, hidden_size=128,
                            intermediate_size=256, num_layers=2, num_heads=2,
                            max_position=128),
}


def _plain(emb: nn.Module) -> bool:
    """Whether an embedding does no more than look up rows of its weight."""
    return _own(emb, nn.Embedding) and emb.max_norm is None


def _first_pays(cu: list) -> bool:
    """Whether the last block is computed for first rows only: three launches more,
    of fewer rows. us of the model (bge-base) with all rows and so: 1 text of 511
    658 and 653, 3 of 400 755 and 746, 64 of 20 719 and 717, 64 of 40 933 and 915,
    64 of 250 3512 and 3322."""
    return cu[-1] >= max(1024, 8 * (len(cu) - 1)) and all(
        b > a for a, b in zip(cu, cu[1:]))


@_written
class BertLayer(nn.Module):
    PARAMS = ("qkv_w", "qkv_b", "attn_out_w", "attn_out_b", "attn_ln_w",
              "attn_ln_b", "up_w", "up_b", "down_w", "down_b", "out_ln_w",
              "out_ln_b")

    def __init__(self, cfg: BertConfig):
        super().__init__()
        h = cfg.hidden_size
        self.qkv_w = nn.Parameter(torch.empty(3 * h, h))
        self.qkv_b = nn.Parameter(torch.zeros(3 * h))
        self.attn_out_w = nn.Parameter(torch.empty(h, h))
        self.attn_out_b = nn.Parameter(torch.zeros(h))
        self.attn_ln_w = nn.Parameter(torch.ones(h))
        self.attn_ln_b = nn.Parameter(torch.zeros(h))
        self.up_w = nn.Parameter(torch.empty(cfg.intermediate_size, h))
        self.up_b = nn.Parameter(torch.zeros(cfg.intermediate_size))
        self.down_w = nn.Parameter(torch.empty(h, cfg.intermediate_size))
        self.down_b = nn.Parameter(torch.zeros(h))
        self.out_ln_w = nn.Parameter(torch.ones(h))
        self.out_ln_b = nn.Parameter(torch.zeros(h))
        self.cfg = cfg
        self.hd = cfg.hidden_size // cfg.num_heads
        self.scale = self.hd ** -0.5

    def first_rows(self, x, cu, max_len):
        """The first row of each text, all of which have tokens, and the
        boundaries of texts of a row each; None where forward is to be asked.
        For a layer that is _own: a hook or a module around it would not see it."""
        if tuple(self._parameters) != self.PARAMS:
            return None
        return ops.text_block_first(x, cu, max_len, self.cfg.num_heads,
                                    self.scale, self.cfg.layer_norm_eps,
                                    list(self._parameters.values()))

    def forward(self, x, cu, max_len):
        if tuple(self._parameters) == self.PARAMS:
            out = ops.text_block(x, cu, max_len, self.cfg.num_heads, self.scale,
                                 self.cfg.layer_norm_eps,
                                 list(self._parameters.values()))
            if out is not None:
                return out
        T = x.shape[0]
        h = self.cfg.hidden_size
        qkv = ops.gemm_bf16(x, self.qkv_w, self.qkv_b)
        nh = self.cfg.num_heads
        q, k, v = (t.view(T, nh, self.hd)
                   for t in qkv.split([h, h, h], dim=-1))
        o = ops.attn_prefill(q, k, v, cu, max_len, self.scale, causal=False)
        a = ops.gemm_bf16(o.view(T, h), self.attn_out_w, self.attn_out_b)
        x = ops.add_layer_norm(x, a, self.attn_ln_w, self.attn_ln_b,
                               self.cfg.layer_norm_eps)
        m = ops.gemm_bf16(x, self.up_w, self.up_b, act=1)   # fused GELU
        m = ops.gemm_bf16(m, self.down_w, self.down_b)
        return ops.add_layer_norm(x, m, self.out_ln_w, self.out_ln_b,
                                  self.cfg.layer_norm_eps)


class BertEmbeddingModel(nn.Module):
    def __init__(self, cfg: BertConfig):
        super().__init__()
        self.cfg = cfg
        self.word_emb = nn.Embedding(cfg.vocab_size, cfg.hidden_size)
        self.pos_emb = nn.Embedding(cfg.max_position, cfg.hidden_size)
        self.emb_ln_w = nn.Parameter(torch.ones(cfg.hidden_size))
        self.emb_ln_b = nn.Parameter(torch.zeros(cfg.hidden_size))
        self.layers = nn.ModuleList(
            [BertLayer(cfg) for _ in range(cfg.num_layers)])

    @torch.inference_mode()
    def forward(self, input_ids: torch.Tensor, cu_seqlens: torch.Tensor,
                max_len: int) -> torch.Tensor:
        """input_ids: [T] varlen concat; returns [B, H] L2-normalized. A text
        longer than the table of places is refused; on GPU an id outside the
        vocabulary, which the host doesn't see, makes its text's result NaN."""
        T = input_ids.shape[0]
        # one read by the host, for the checks and the mean's bounds
        cu = cu_seqlens.tolist()
        if cu[0] != 0 or cu[-1] != T or any(
                b < a for a, b in zip(cu, cu[1:])):
            raise ValueError(f"boundaries {cu} do not cut {T} tokens")
        if self.cfg.pooling != "mean" and cu[-2] == T:
            raise IndexError("a last text without tokens")
        if _plain(self.pos_emb):
            places = self.pos_emb.weight.shape[0]
            if any(b - a > places for a, b in zip(cu, cu[1:])):
                raise IndexError(f"a text of more than {places} tokens")
        x = None
        if _plain(self.word_emb) and _plain(self.pos_emb):
            x = ops.text_embed(input_ids, cu_seqlens, self.word_emb.weight,
                               self.pos_emb.weight, self.emb_ln_w,
                               self.emb_ln_b, self.cfg.layer_norm_eps)
        if x is None:
            positions = torch.arange(T, device=input_ids.device) - \
                torch.repeat_interleave(cu_seqlens[:-1].long(),
                                        cu_seqlens.diff(), output_size=T)
            x = self.word_emb(input_ids) + self.pos_emb(positions)
            x = ops.layer_norm(x, self.emb_ln_w, self.emb_ln_b,
                               self.cfg.layer_norm_eps)
        last = len(self.layers) - 1
        for i, layer in enumerate(self.layers):
            if i == last and self.cfg.pooling != "mean" and \
                    _own(layer, BertLayer) and _first_pays(cu):
                first = layer.first_rows(x, cu_seqlens, max_len)
                if first is not None:
                    emb = ops.text_pool(*first)
                    if emb is not None:
                        return emb
            x = layer(x, cu_seqlens, max_len)
        if self.cfg.pooling == "mean":
            emb = torch.stack([x[s:e].float().mean(0)
                               for s, e in zip(cu, cu[1:])])
        else:
            emb = ops.text_pool(x, cu_seqlens)
            if emb is not None:
                return emb
            emb = x[cu_seqlens[:-1].long()].float()
        return torch.nn.functional.normalize(emb, dim=-1)

    @torch.inference_mode()
    def init_random(self, seed: int = 0):
        on_gpu = next(self.parameters()).is_cuda
        if on_gpu:
            torch.cuda.manual_seed(seed)
        g = None if on_gpu else torch.Generator().manual_seed(seed)
        for name, p in self.named_parameters():
            if name.endswith(("_b", "ln_w", "ln_b")):
                continue  # keep zeros/ones defaults
            if on_gpu:
                p.data.normal_(0.0, 0.02)
            else:
                t = torch.empty(p.shape, dtype=torch.float32)
                t.normal_(0.0, 0.02, generator=g)
                p.data.copy_(t.to(p.dtype))
        return self

    def memory_bytes(self) -> int:
        return sum(p.numel() * p.element_size() for p in self.parameters())
