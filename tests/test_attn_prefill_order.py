"""Prompt attention: which workgroup has which queries, waves without any, and a
maximum that moves from tile to tile, against 64 bits. Weights and results are
rounded to bf16, by at most 2^-8 of each: a result is at most 2^-8 of the weighted sum
of its values' sizes, and 2^-8 of itself, from the exact one; a tenth of that is left
to exponentials and sums in 32 bits."""
import pytest
import torch

import helix_amd.ops as ops

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _check(lens, hq, hkv, d, causal, q, k, v, scale):
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(),
                      dtype=torch.int32, device=DEV)
    got = ops.attn_prefill(q, k, v, cu, max(lens), scale, causal).double()
    want, sizes = torch.empty_like(got), torch.empty_like(got)
    for a, b in zip(cu.tolist(), cu.tolist()[1:]):
        x, y, z = (t[a:b].double().transpose(0, 1).contiguous()
                   for t in (q, k, v))
        y, z = (t.repeat_interleave(hq // hkv, 0) for t in (y, z))
        s = x @ y.transpose(1, 2).contiguous() * scale
        if causal:
            s.masked_fill_(torch.ones(b - a, b - a, dtype=torch.bool,
                                      device=DEV).triu(1), -torch.inf)
        p = s.softmax(-1)
        want[a:b] = (p @ z).transpose(0, 1)
        sizes[a:b] = (p @ z.abs()).transpose(0, 1)
    assert ((got - want).abs()
            <= 1.1 * 2 ** -8 * (sizes + want.abs())).all()


# groups of heads: fewer than XCDs, a multiple of them, many that are none; texts
# of one query, of a wave, a workgroup and one more
@pytest.mark.parametrize("lens,hq,hkv,d,causal", [
    ([5], 4, 2, 64, False), ([300, 1, 129], 12, 12, 64, False),
    ([32, 33, 97], 16, 1, 128, True), ([288] * 8, 16, 16, 64, False),
    ([1, 500, 64, 31, 160, 128, 255], 28, 4, 128, True),
    ([77, 20, 410], 12, 12, 64, True), ([1000], 32, 8, 128, True),
    ([640, 2], 28, 4, 128, False)])
def test_places(lens, hq, hkv, d, causal):
    g = torch.Generator(device=DEV).manual_seed(sum(lens))
    q, k, v = (torch.randn(sum(lens), n, d, device=DEV, generator=g).bfloat16()
               for n in (hq, hkv, hkv))
    _check(lens, hq, hkv, d, causal, q, k, v, d ** -0.5)


# scores that rise or fall from tile to tile by this much of log2 of a weight
@pytest.mark.parametrize("rise", [0.5, 3.0, 8.0, 30.0, -5.0])
@pytest.mark.parametrize("d,causal", [(64, False), (128, True)])
def test_rising_scores(rise, d, causal):
    g = torch.Generator(device=DEV).manual_seed(7)
    n, h = 700, 8
    q, k, v = (torch.randn(n, h, d, device=DEV, generator=g) for _ in range(3))
    # the first element alone carries the rise; a row's own level differs
    q[..., 0] = 1.0
    at = torch.arange(n, device=DEV) // 64
    k[..., 0] = (at * rise * 0.6931 * d ** 0.5)[:, None]
    _check([n], h, h, d, causal, q.bfloat16(), k.bfloat16(), v.bfloat16(),
           d ** -0.5)


# whole rounds of groups and some left over, which are cut into heads: fewer heads
# than XCDs, more, and seven groups
@pytest.mark.parametrize("lens,hq,hkv,d,causal", [
    ([128] * 9, 28, 4, 128, True), ([130, 1, 40] * 11, 8, 1, 128, True),
    ([33, 200, 129] * 7, 6, 3, 64, False), ([70] * 35, 4, 1, 64, True),
    ([140, 20, 7, 129, 260] * 2 + [64], 14, 7, 64, False),
    ([150] * 41, 2, 1, 64, True)])
def test_groups_left_over(lens, hq, hkv, d, causal):
    g = torch.Generator(device=DEV).manual_seed(len(lens))
    q, k, v = (torch.randn(sum(lens), n, d, device=DEV, generator=g).bfloat16()
               for n in (hq, hkv, hkv))
    _check(lens, hq, hkv, d, causal, q, k, v, d ** -0.5)


@pytest.mark.parametrize("texts", [32767, 32768])
def test_more_rounds_than_a_grid_has_along_y(texts):
    """Of one key, a result is its value."""
    q, k, v = (torch.randn(texts, 16, 64, device=DEV).bfloat16()
               for _ in range(3))
    cu = torch.arange(texts + 1, dtype=torch.int32, device=DEV)
    assert torch.equal(ops.attn_prefill(q, k, v, cu, 1, 0.125, False), v)
