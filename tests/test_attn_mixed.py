"""Replies and prompt portions in one launch give the bits of a launch each."""
import pytest
import torch

import helix_amd.ops as ops

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _inputs(hq, hkv, d, bs, fp8, lens, new, cached):
    g = torch.Generator(device=DEV).manual_seed(len(lens) + sum(new))
    r = lambda *s: torch.randn(*s, device=DEV, generator=g).bfloat16()  # noqa: E731
    pages = [-(-n // bs) for n in lens]
    caches = [r(sum(pages) + 1, hkv, bs, d) for _ in range(2)]
    if fp8:
        caches = [ops.kv_fp8_quant(c) for c in caches]
    bt = torch.zeros(len(lens), max(pages), dtype=torch.int32)
    order = torch.randperm(sum(pages)).tolist()
    for i, n in enumerate(pages):
        bt[i, :n] = torch.tensor([order.pop() for _ in range(n)])
    cu = [torch.tensor([0] + torch.tensor(x).cumsum(0).tolist(),
                       dtype=torch.int32, device=DEV)
          for x in (new, [a + b for a, b in zip(new, cached)])]
    keys = sum(new) + sum(cached)
    return (r(sum(new), hq, d), r(keys, hkv, d), r(keys, hkv, d), *cu,
            max(new)), (r(len(lens), hq, d), *caches, bt.to(DEV),
                        torch.tensor(lens, dtype=torch.int32, device=DEV))


# fewer workgroups than places and more, cut sequences and whole ones, a reply
# without keys, windows
@pytest.mark.parametrize("hq,hkv,d,bs,fp8,lens,new,cached,window", [
    (32, 8, 128, 16, False, [1], [17], [0], 0),
    (32, 8, 128, 16, False, [3000, 1, 700, 0, 129], [130, 1], [500, 33], 0),
    (32, 8, 128, 16, True, [900, 4100, 64], [700], [1200], 512),
    (8, 1, 128, 8, False, [2000] * 40, [257, 128, 3], [0, 0, 900], 0),
    (64, 8, 128, 32, True, [40, 500], [1000], [0], 300)])
def test_same_bits(hq, hkv, d, bs, fp8, lens, new, cached, window):
    (qp, k, v, cu, cuk, most), (qd, kc, vc, bt, sl) = _inputs(
        hq, hkv, d, bs, fp8, lens, new, cached)
    s, hi, B = d ** -0.5, max(lens), len(lens)
    ws = ops.decode_workspace(B, hq, d, hi, DEV)
    op, od = torch.full_like(qp, 7.0), torch.full_like(qd, 7.0)
    assert ops.mixed_attention((op, qp, k, v, cu, cuk, most),
                               (od, qd, kc, vc, bt, sl, *ws, hi), s, window)
    want = ops.paged_attn_decode(qd, kc, vc, bt, sl, s, ws, hi, window)
    assert torch.equal(od, want)
    assert torch.equal(op, ops.attn_prefill(qp, k, v, cu, most, s, True,
                                            window, cuk))


@pytest.mark.parametrize("hq,hkv,d,bs", [(8, 2, 64, 16), (8, 4, 128, 16),
                                         (8, 2, 128, 24), (8, 2, 128, 4)])
def test_left_alone(hq, hkv, d, bs):
    (qp, k, v, cu, cuk, most), (qd, kc, vc, bt, sl) = _inputs(
        hq, hkv, d, bs, False, [50, 9], [20], [0])
    ws = ops.decode_workspace(2, hq, d, 50, DEV)
    op, od = torch.full_like(qp, 7.0), torch.full_like(qd, 7.0)
    assert not ops.mixed_attention((op, qp, k, v, cu, cuk, most),
                                   (od, qd, kc, vc, bt, sl, *ws, 50), 0.1, 0)
    assert (op == 7).all() and (od == 7).all()


# many short replies leave the joint launch to portions that hide more than they lose
@pytest.mark.parametrize("rows,bound,fp8,new,cached,joint", [
    (230, 300, True, [17], [0], True), (256, 300, True, [17], [0], False),
    (256, 300, True, [17], [100], True), (512, 300, True, [300], [0], False),
    (512, 300, True, [17], [700], True), (256, 1025, True, [17], [0], True),
    (512, 300, False, [17], [0], False), (512, 385, False, [17], [0], True),
    (512, 300, False, [17], [100], True), (450, 300, False, [17], [0], True)])
def test_where_one_launch_pays(rows, bound, fp8, new, cached, joint):
    """Either way the model's step has the same bits: what is declined is done by
    the two launches."""
    lens = [bound] + [1 + 37 * i % 40 for i in range(1, rows)]
    (qp, k, v, cu, cuk, most), (qd, kc, vc, bt, sl) = _inputs(
        32, 8, 128, 16, fp8, lens, new, cached)
    ws = ops.decode_workspace(rows, 32, 128, bound, DEV)
    op, od = torch.full_like(qp, 7.0), torch.full_like(qd, 7.0)
    assert joint == ops.mixed_attention(
        (op, qp, k, v, cu, cuk, most), (od, qd, kc, vc, bt, sl, *ws, bound),
        0.1, 0)
    if joint:
        assert torch.equal(od, ops.paged_attn_decode(qd, kc, vc, bt, sl, 0.1,
                                                     ws, bound))
        assert torch.equal(op, ops.attn_prefill(qp, k, v, cu, most, 0.1, True,
                                                0, cuk))
    else:
        assert (op == 7).all() and (od == 7).all()
