"""How a layer's launches of a few rows are put together: with stand-ins for them on
the CPU, the model gives what it gives without."""
import pytest
import torch
import torch.nn.functional as F

from helix_amd import ops
from helix_amd.models.llama import PRESETS, LlamaForCausalLM
from helix_amd.models.meta import PrefillMeta


def _normed(x):
    if not isinstance(x, ops.Unscaled):
        return x
    mean = x.squares.sum(1, keepdim=True) / x.rows.shape[1]
    return x.rows * torch.rsqrt(mean + x.eps)


def _join(x, w, residual, norm_w, eps):
    residual += F.linear(x, w)
    return ops.Unscaled(residual * norm_w,
                        residual.square().sum(1, keepdim=True), eps)


def _glu(x, w):
    g, u = F.linear(_normed(x), w).chunk(2, 1)
    return F.silu(g) * u


def _qkv(positions, x, w, bias, *heads):
    return ops.rope_qkv_cache(positions, F.linear(_normed(x), w, bias), *heads)


def _pass(model, n=9):
    cfg = model.cfg
    caches = [tuple(torch.zeros(1, cfg.num_kv_heads, 16, cfg.head_dim)
                    for _ in range(2)) for _ in range(cfg.num_layers)]
    meta = PrefillMeta(cu_seqlens=torch.tensor([0, n], dtype=torch.int32),
                       max_seqlen=n, slot_mapping=torch.arange(n),
                       positions=torch.arange(n))
    return model(torch.arange(n) * 3, caches, meta), caches


@pytest.mark.parametrize("preset", ["tiny-gqa", "tiny-qwen"])
@pytest.mark.parametrize("other", [[], [0], [2], [0, 1, 2, 3]])
def test_layers_of_a_few_rows(monkeypatch, preset, other):
    """Norms of layers with weights and eps of their own, beside layers (other)
    that go the long way."""
    model = LlamaForCausalLM(PRESETS[preset]).init_random(3)
    for i, layer in enumerate(model.layers):
        layer.eps = (1e-5, 0.3, 2.0, 0.01)[i]
        for w in (layer.input_norm_w, layer.post_norm_w):
            w.data += 0.3 * torch.randn_like(w)
    want, kept = _pass(model)
    for name, f in (("layer_rows_fit", lambda *a: True),
                    ("_bias_fits", lambda *a: True), ("rows_join", _join),
                    ("rows_glu", _glu), ("rows_qkv", _qkv)):
        monkeypatch.setattr(ops, name, f)
    for i in other:
        if i < len(model.layers):
            model.layers[i].register_forward_hook(lambda m, i, o: None)
    got, caches = _pass(model)
    torch.testing.assert_close(got, want, atol=1e-5, rtol=1e-5)
    for a, b in zip(kept, caches):
        for x, y in zip(a, b):
            torch.testing.assert_close(x, y, atol=1e-5, rtol=1e-5)


def test_a_layer_is_asked_shortly_before_its_turn(monkeypatch):
    """What a layer's launches may be is asked while those of the layer before are
    under way, not of all layers before the first."""
    from helix_amd.models.llama import DecoderLayer
    model = LlamaForCausalLM(PRESETS["tiny-gqa"]).init_random(3)
    for name, f in (("layer_rows_fit", lambda *a: True), ("rows_join", _join),
                    ("rows_glu", _glu), ("rows_qkv", _qkv)):
        monkeypatch.setattr(ops, name, f)
    order, few = [], DecoderLayer.few

    def asked(self, x):
        order.append(("few", list(model.layers).index(self)))
        return few(self, x)

    monkeypatch.setattr(DecoderLayer, "few", asked)
    glu = ops.rows_glu
    monkeypatch.setattr(ops, "rows_glu", lambda *a: order.append(
        ("run", sum(k == "run" for k, _ in order))) or glu(*a))
    _pass(model)
    assert order == [("few", 0), ("few", 1), ("run", 0), ("few", 2),
                     ("run", 1), ("few", 3), ("run", 2), ("run", 3)]
