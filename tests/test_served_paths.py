"""Ways that models take through their launches on the GPU, each against the other way
of the same model: replies and portions in one launch or two, rows that are asked for,
layers of a few rows, first rows of texts."""
from dataclasses import replace

import pytest
import torch

from helix_amd import ops
from helix_amd.engine.engine import EngineConfig, LLMEngine
from helix_amd.models import bert
from helix_amd.models.llama import DecoderLayer, LlamaConfig, LlamaForCausalLM

pytestmark = pytest.mark.gpu

CFG = LlamaConfig(name="two layers", vocab_size=1024, hidden_size=1024,
                  intermediate_size=2048, num_layers=2, num_heads=8,
                  num_kv_heads=2, head_dim=128, max_position=4096)


def _engine(weights=None, cache="bf16", **cfg):
    model = LlamaForCausalLM(replace(CFG, **cfg)).bfloat16().cuda()
    g = torch.Generator(device="cuda").manual_seed(11)
    for name, p in model.named_parameters():
        p.data.normal_(0.0, 1.0 if name.startswith("embed") else 0.02,
                       generator=g)
        if name.endswith("norm_w"):
            p.data += 1.0
    return LLMEngine(EngineConfig(
        model="tiny", max_num_seqs=64, max_model_len=4096,
        kv_cache_blocks=1024, eos_token_id=-1, quantization=weights,
        kv_cache_dtype=cache, mixed_steps=True), "cuda", model=model)


def _ids(n, seed):
    return torch.randint(0, 1024, (n,), generator=torch.Generator()
                         .manual_seed(seed)).tolist()


def _step(eng, replies, portions, every=False):
    """Scores of a step: replies to sequences of these lengths beside portions of
    (cached, new) tokens, at their last or at every place."""
    entries = []
    for i, n in enumerate(replies):
        eng.extend([(f"r{i}", _ids(n, i), [])])
        entries.append((f"r{i}", [i], [0]))
    for i, (cached, new) in enumerate(portions):
        if cached:
            eng.extend([(f"p{i}", _ids(cached, 100 + i), [])])
        entries.append((f"p{i}", _ids(new, 200 + i),
                        list(range(new)) if every else [new - 1]))
    out = eng.extend(entries)
    for sid, _, _ in entries:
        eng.release(sid)
    return out.float()


# fresh and cached portions; a workspace for 64 sequences of 4096 throughout
@pytest.mark.parametrize("cache", ["bf16", "fp8"])
@pytest.mark.parametrize("window", [0, 300])
@pytest.mark.parametrize("replies,portions", [
    ([5, 700, 64], [(0, 33)]), ([1500, 20], [(500, 200), (16, 3)]),
    ([30] * 20, [(0, 300), (0, 17)])])
def test_mixed_step_in_one_launch(monkeypatch, cache, window, replies,
                                  portions):
    """The same bits as in two."""
    eng, took = _engine(cache=cache, sliding_window=window), []
    one = ops.mixed_attention
    monkeypatch.setattr(ops, "mixed_attention",
                        lambda *a: took.append(one(*a)) or took[-1])
    got = _step(eng, replies, portions)
    assert took == [True, True]                 # layers
    monkeypatch.setattr(ops, "mixed_attention", lambda *a: False)
    assert torch.equal(got, _step(eng, replies, portions))


# bf16: two orders of the same sums in the last layer, five products and sums round
# 2^-9 each. 8-bit rows: what moves by 2^-8 is rounded to another byte, 2^-3 away, in a
# share of 2^-5: 2^-3 2^-2.5 of a product, twice in the layer
@pytest.mark.parametrize("weights,near", [(None, 5 * 2 ** -9),
                                          ("fp8", 2 * 2 ** -5.5)])
@pytest.mark.parametrize("replies,portions", [
    ([], [(0, 256)]), ([], [(0, 300), (0, 41)]), ([], [(200, 400)]),
    ([700, 5, 64], [(500, 300)]), ([9] * 40, [(0, 260), (0, 17)])])
def test_rows_asked_for(monkeypatch, weights, near, replies, portions):
    eng = _engine(weights)
    some, seen = eng.model._hidden, []

    def hidden(*a):
        seen.append(len(a) > 3 and a[3] is not None)
        return some(*a)

    monkeypatch.setattr(eng.model, "_hidden", hidden)
    got = _step(eng, replies, portions)
    assert seen[-1]
    monkeypatch.setattr(DecoderLayer, "unseen", lambda self: False)
    want = _step(eng, replies, portions)
    assert not seen[-1] and got.shape == want.shape
    assert (got - want).norm() < near * want.norm()
    assert ((got - want).norm(dim=1) < 2 * near * want.norm(dim=1)).all()


# rows go to a product before they are divided by their root: another order of the
# roundings of the norm, the products and the sums of both layers, 2^-9 each
@pytest.mark.parametrize("cache", ["bf16", "fp8"])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("replies,portions", [
    ([40], []), ([5, 700, 64, 16], []), ([300] * 16, []), ([], [(0, 13)]),
    ([], [(100, 7), (0, 5)]), ([90, 4], [(0, 9)])])
def test_layers_of_a_few_rows(monkeypatch, cache, bias, replies, portions):
    few, fits = _engine(cache=cache, attention_bias=bias), []
    fit = ops.layer_rows_fit
    monkeypatch.setattr(ops, "layer_rows_fit",
                        lambda *a: fits.append(fit(*a)) or fits[-1])
    got = _step(few, replies, portions, every=True)
    assert fits and fits[-1]
    monkeypatch.setattr(ops, "layer_rows_fit", lambda *a: False)
    want = _step(_engine(cache=cache, attention_bias=bias), replies, portions,
                 every=True)
    # pages that hold 8 bits differ where a key falls on another side
    near = (12 if cache == "bf16" else 24) * 2 ** -9
    assert (got - want).norm() < near * want.norm()


@pytest.mark.parametrize("lens", [[512, 512], [20, 1, 500, 77, 426],
                                  [16] * 100])
def test_first_rows_of_the_text_encoder(monkeypatch, lens):
    """Two ways through its last block, five products and sums of 2^-9 each; a
    text's is its own."""
    cfg = replace(bert.BERT_PRESETS["tiny-bert"], max_position=512)
    model = bert.BertEmbeddingModel(cfg).init_random(5).bfloat16().cuda()
    for layer in model.layers:
        for p in layer.parameters():
            if p.dim() == 2:
                p.data.mul_(4.0)               # a spread of 0.08
    n = sum(lens)
    ids = torch.randint(0, 512, (n,), device="cuda",
                        generator=torch.Generator("cuda").manual_seed(n))
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(),
                      dtype=torch.int32, device="cuda")
    asked, first = [], ops.text_block_first
    monkeypatch.setattr(ops, "text_block_first",
                        lambda *a: asked.append(first(*a)) or asked[-1])
    got = model(ids, cu, max(lens))
    assert len(asked) == 1 and asked[0] is not None
    monkeypatch.setattr(bert, "_first_pays", lambda cu: False)
    want = model(ids, cu, max(lens))
    assert len(asked) == 1
    assert ((got - want).norm(dim=1) < 5 * 2 ** -9).all()     # of length 1
    assert (got @ want.T).argmax(1).tolist() == list(range(len(lens)))
