"""Rows of a prompt that nobody asks for leave before the last layer's feed-forward:
those asked for are what a pass over all rows gives, and hooks see all of them."""
import pytest
import torch

from helix_amd.models.llama import PRESETS, LlamaForCausalLM
from helix_amd.models.meta import PrefillMeta


def _step(lens):
    T = sum(lens)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(),
                      dtype=torch.int32)
    pos = torch.cat([torch.arange(n) for n in lens])
    return torch.arange(T) % 500, PrefillMeta(
        cu_seqlens=cu, max_seqlen=max(lens),
        slot_mapping=torch.arange(T), positions=pos)


def _caches(cfg, T):
    n = -(-T // 16)
    return [(torch.zeros(n, cfg.num_kv_heads, 16, cfg.head_dim),
             torch.zeros(n, cfg.num_kv_heads, 16, cfg.head_dim))
            for _ in range(cfg.num_layers)]


# too few tokens, one row, several, more than half
@pytest.mark.parametrize("lens,rows", [
    ([200], [199]), ([256], [255]), ([300, 40], [299, 339, 7]),
    ([256], list(range(129))), ([256], list(range(0, 256, 2)))])
def test_same_rows(lens, rows):
    cfg = PRESETS["tiny"]
    model = LlamaForCausalLM(cfg).init_random(3)
    ids, meta = _step(lens)
    a, b = _caches(cfg, sum(lens)), _caches(cfg, sum(lens))
    want = model(ids, a, meta)[torch.tensor(rows)]
    got = model.forward_rows(ids, b, meta, torch.tensor(rows))
    # sums of the products in another order: fp32
    torch.testing.assert_close(got, want, atol=1e-5, rtol=1e-5)
    for (k, v), (x, y) in zip(a, b):
        assert torch.equal(k, x) and torch.equal(v, y)


@pytest.mark.parametrize("where", [
    "layers.1", "layers.1.attn.o_proj", "layers.1.mlp.down_proj", ""])
def test_hooks_see_all(where):
    model = LlamaForCausalLM(PRESETS["tiny"]).init_random(3)
    seen = []
    model.get_submodule(where).register_forward_hook(
        lambda m, i, o: seen.append((o[0] if isinstance(o, tuple)
                                     else o).shape[0]))
    ids, meta = _step([300])
    out = model.forward_rows(ids, _caches(model.cfg, 300), meta,
                             torch.tensor([299]))
    assert seen == [300] and out.shape[0] == 1


@pytest.mark.gpu
@pytest.mark.parametrize("lens,h,inner,heads", [
    ([1], 128, 256, 2), ([20, 1, 44, 500], 768, 3072, 12),
    ([64] * 70, 256, 512, 2), ([300, 129], 1024, 4096, 8)])
def test_first_rows_of_texts(lens, h, inner, heads):
    """Two ways through a block round what five products and sums of unit spread
    give to bf16, 2^-9 of it in the mean each."""
    from helix_amd import ops
    torch.manual_seed(len(lens))
    r = lambda *s, std=1.0: (torch.randn(*s, device="cuda") * std).bfloat16()  # noqa: E731
    p = [r(3 * h, h, std=h ** -0.5), r(3 * h, std=0.3), r(h, h, std=h ** -0.5),
         r(h, std=0.3), 1 + r(h, std=0.1), r(h, std=0.1),
         r(inner, h, std=h ** -0.5), r(inner, std=0.3),
         r(h, inner, std=inner ** -0.5), r(h, std=0.3), 1 + r(h, std=0.1),
         r(h, std=0.1)]
    x = r(sum(lens), h)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(),
                      dtype=torch.int32, device="cuda")
    with torch.inference_mode():
        args = (x, cu, max(lens), heads, (h // heads) ** -0.5, 1e-12, p)
        want = ops.text_block(*args)[cu[:-1].long()].float()
        got, starts = ops.text_block_first(*args)
    assert starts.tolist() == list(range(len(lens) + 1))
    assert ((got.float() - want).norm() / want.norm()).item() < 5 * 2 ** -9


class Delegating(torch.nn.Module):
    """A wrapper in the manner of adapters: a forward of its own, every other
    attribute the inner module's."""

    def __init__(self, inner, add=0.0):
        super().__init__()
        self.inner, self.add, self.calls = inner, add, 0

    def __getattr__(self, name):
        try:
            return super().__getattr__(name)
        except AttributeError:
            return getattr(super().__getattr__("inner"), name)

    def forward(self, *args):
        self.calls += 1
        out = self.inner(*args)
        return (out[0] + self.add, *out[1:]) if isinstance(out, tuple) \
            else out + self.add


class Plain(torch.nn.Module):
    """A layer in place of the model's with nothing but a forward."""

    def __init__(self, inner):
        super().__init__()
        self.inner = inner

    def forward(self, *args):
        return self.inner(*args)


def _engine(model):
    from helix_amd.engine.engine import EngineConfig, LLMEngine
    return LLMEngine(EngineConfig(model="tiny", max_num_seqs=4,
                                  max_model_len=512, kv_cache_blocks=64,
                                  eos_token_id=-1), "cpu", model=model)


def _last_scores(eng, n):
    """Scores behind the last of n tokens, through the engine's step."""
    return eng.extend([("a", [t % 500 for t in range(n)], [n - 1])])


WRAPPERS = {"plain": Plain, "delegating": Delegating,
            "compiled": lambda m: torch.compile(m, backend="eager")}


@pytest.mark.parametrize("wrap", list(WRAPPERS))
@pytest.mark.parametrize("n", [200, 300])
def test_other_last_layer(wrap, n):
    """It gets and gives all rows, and the scores are those asked for."""
    model = LlamaForCausalLM(PRESETS["tiny"]).init_random(3)
    ids, meta = _step([n])
    want = model.compute_logits(model(ids, _caches(model.cfg, n),
                                      meta)[n - 1:])
    model.layers[-1] = WRAPPERS[wrap](model.layers[-1])
    got = _last_scores(_engine(model), n)
    assert got.shape == want.shape
    torch.testing.assert_close(got, want, atol=1e-5, rtol=1e-5)


@pytest.mark.parametrize("wrap", ["delegating", "compiled"])
@pytest.mark.parametrize("n", [200, 300])
def test_other_model(wrap, n):
    """A wrapper around the whole model is what the engine calls."""
    model = LlamaForCausalLM(PRESETS["tiny"]).init_random(3)
    ids, meta = _step([n])
    hidden = model(ids, _caches(model.cfg, n), meta)[n - 1:]
    eng = _engine(model)
    if wrap == "compiled":
        graphs = []
        eng.model = torch.compile(
            model, backend=lambda g, _: graphs.append(g) or g.forward)
        add = 0.0
    else:
        eng.model = Delegating(model, add=0.25)
        add = 0.25
    got = _last_scores(eng, n)
    assert graphs if wrap == "compiled" else eng.model.calls == 1
    torch.testing.assert_close(got, model.compute_logits(hidden + add),
                               atol=1e-5, rtol=1e-5)


@pytest.mark.parametrize("wrap", list(WRAPPERS))
@pytest.mark.parametrize("pooling", ["cls", "mean"])
def test_other_last_layer_of_texts(monkeypatch, wrap, pooling):
    """The text encoder's: its forward is called, with all rows. First rows alone
    are computed on the GPU; a stand-in counts who asks for them."""
    from dataclasses import replace
    from helix_amd import ops
    from helix_amd.models.bert import BERT_PRESETS, BertEmbeddingModel
    asked = []
    monkeypatch.setattr(ops, "text_block_first",
                        lambda x, *a: asked.append(x.shape[0]))
    model = BertEmbeddingModel(replace(BERT_PRESETS["tiny-bert"],
                                       pooling=pooling)).init_random(5)
    cu = torch.arange(0, 1281, 128, dtype=torch.int32)
    ids = torch.arange(1280) % 500
    want = model(ids, cu, 128)
    assert asked == ([1280] if pooling == "cls" else [])
    model.layers[-1] = WRAPPERS[wrap](model.layers[-1])
    torch.testing.assert_close(model(ids, cu, 128), want, atol=1e-5, rtol=1e-5)
    assert asked == ([1280] if pooling == "cls" else [])
    if wrap == "delegating":
        assert model.layers[-1].calls == 1


@pytest.mark.gpu
@pytest.mark.parametrize("lens", [[0, 40, 0, 0, 7, 0], [0, 0], [1]])
def test_first_rows_of_texts_without_tokens(lens):
    """Of a text without tokens, the last one too, there is no row: NaN, and
    nothing behind the rows is read. The others as above."""
    from helix_amd.models.bert import BERT_PRESETS, BertEmbeddingModel
    layer = BertEmbeddingModel(BERT_PRESETS["tiny-bert"]).init_random(
        5).bfloat16().cuda().layers[0]
    x = torch.randn(max(sum(lens), 1), 128).bfloat16().cuda()
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(),
                      dtype=torch.int32, device="cuda")
    full = [i for i, n in enumerate(lens) if n]
    with torch.inference_mode():
        want = layer(x, cu, max(lens))[cu[full].long()].float()
        got, starts = layer.first_rows(x, cu, max(lens))
    assert starts.tolist() == list(range(len(lens) + 1))
    assert got[[i for i, n in enumerate(lens) if not n]].isnan().all()
    assert (got[full].float() - want).norm() <= 5 * 2 ** -9 * want.norm()


def _mixed(model, monkeypatch):
    """Scores of a step with a reply and a portion, and how often both were to be
    attended in one launch (the CPU declines)."""
    from helix_amd import ops
    eng, asked = _engine(model), []
    monkeypatch.setattr(ops, "mixed_attention",
                        lambda *a: asked.append(a) is not None)
    w = eng.decode_ws = eng.decode_ws or (torch.zeros(4, 4, 4, 64),
                                          torch.zeros(4, 4, 4, 2))
    assert len(w) == 2
    eng.extend([("a", list(range(20)), [19])])
    return eng.extend([("a", [7], [0]), ("b", list(range(30)), [29])]), \
        len(asked)


@pytest.mark.parametrize("which", ["_attend_decode", "_attend_prefill"])
@pytest.mark.parametrize("where", ["class", "instance"])
def test_attention_of_its_own_in_mixed_steps(monkeypatch, which, where):
    """An Attention with another way to attend is asked for it in mixed steps."""
    from helix_amd.models.llama import Attention
    make = lambda: LlamaForCausalLM(PRESETS["tiny"]).init_random(3)  # noqa: E731
    want, asked = _mixed(make(), monkeypatch)
    assert asked == 2                           # layers
    model, calls = make(), []
    attn = model.layers[0].attn
    base = getattr(Attention, which)

    def other(self, *args):
        calls.append(args)
        return base(self, *args)

    if where == "class":
        attn.__class__ = type("Other", (Attention,), {which: other})
    else:
        setattr(attn, which, other.__get__(attn))
    got, asked = _mixed(model, monkeypatch)
    assert asked == 1 and len(calls) == (1 if which == "_attend_decode" else 2)
    if which == "_attend_prefill":
        assert calls[1][1] is not None          # a fresh portion's keys
    torch.testing.assert_close(got, want, atol=1e-5, rtol=1e-5)


@pytest.mark.parametrize("kind", ["LlamaForCausalLM", "DecoderLayer",
                                  "Attention", "MLP", "HLinear"])
def test_forward_of_a_class_put_in_place(monkeypatch, kind):
    """It is called for prompts of any length, as often and with as many rows."""
    from helix_amd.models import llama
    cls = getattr(llama, kind)
    base, seen = cls.forward, []

    def forward(self, x, *args):
        seen.append(x.shape[0])
        return base(self, x, *args)

    model = LlamaForCausalLM(PRESETS["tiny"]).init_random(3)
    want = _last_scores(_engine(model), 300)
    monkeypatch.setattr(cls, "forward", forward)
    got = _last_scores(_engine(model), 300)
    rows = {"LlamaForCausalLM": [300], "HLinear": [300] * 8 + [1]}
    assert seen == rows.get(kind, [300] * 2)
    torch.testing.assert_close(got, want, atol=1e-5, rtol=1e-5)
