"""Decode attention on either side of where rows stop being cut."""
import pytest
import torch

from helix_amd import ops
from helix_amd.ops import ref

DEV = "cuda"


@pytest.mark.gpu
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("hq,hkv,d,rows", [
    (8, 2, 64, 1), (8, 2, 64, 63), (8, 2, 64, 64),
    (8, 1, 128, 3), (8, 1, 128, 128), (3, 3, 64, 43)])
@pytest.mark.parametrize("bound", [512, 513, 1024, 1025])
def test_bounds(hq, hkv, d, rows, bound, fp8):
    check(hq, hkv, d, rows, bound, fp8)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [255, 256])
@pytest.mark.parametrize("bound", [2048, 2049])
def test_many(rows, bound):
    check(8, 8, 64, rows, bound, False)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [65535, 65536])
def test_more_rows_than_a_grid_has_along_y(rows):
    """Of one key, a row's result is its value."""
    kc, vc = (torch.randn(3, 2, 8, 64).bfloat16().to(DEV) for _ in range(2))
    bt = (torch.arange(rows) % 3).int()[:, None].to(DEV)
    got = ops.paged_attn_decode(
        torch.randn(rows, 2, 64).bfloat16().to(DEV), kc, vc, bt,
        torch.ones(rows, dtype=torch.int32, device=DEV), 0.125, max_len=1)
    assert torch.equal(got, vc[bt[:, 0].long(), :, 0])


def check(hq, hkv, d, rows, bound, fp8):
    """Lengths from nothing to the bound, heads of a row on every XCD; caches end
    with the last page, and what lies behind a row's end is not a number."""
    torch.manual_seed(rows + bound)
    bs = 16
    lens = [bound] + [(0, 1, 33, 127 + 3 * i, bound - i)[i % 5] if i < 15
                      else 1 + 37 * i % 200 for i in range(1, rows)]
    need = [-(-n // bs) for n in lens]
    q = torch.randn(rows, hq, d, dtype=torch.bfloat16)
    kc = torch.randn(sum(need), hkv, bs, d, dtype=torch.bfloat16)
    vc = torch.randn_like(kc)
    bt = torch.zeros(rows, max(need), dtype=torch.int32)
    for b, pages in enumerate(torch.randperm(sum(need)).int().split(need)):
        bt[b, :need[b]] = pages
    seq_lens = torch.tensor(lens, dtype=torch.int32)
    if fp8:
        kc, vc = ops.kv_fp8_quant(kc), ops.kv_fp8_quant(vc)
    full = [b for b in range(rows) if lens[b]]
    want = torch.zeros(rows, hq, d)
    want[full] = ref.paged_attn_decode(
        q[full].float(), *((ops.kv_fp8_dequant(t) if fp8 else t).float()
                           for t in (kc, vc)), bt[full], seq_lens[full],
        d ** -0.5)
    for b, n in enumerate(lens):
        if n % bs:
            for t in (kc, vc):
                t[bt[b, need[b] - 1].long(), :, n % bs:] = \
                    0x7f if fp8 else float("nan")
    got = ops.paged_attn_decode(q.to(DEV), kc.to(DEV), vc.to(DEV), bt.to(DEV),
                                seq_lens.to(DEV), d ** -0.5, max_len=bound)
    # results rounded to bf16 (half of 2^-7 of a value at most, 2^-8); sums of 32
    # bits over up to 2049 values of weights that add up to 1
    torch.testing.assert_close(got.float().cpu(), want, rtol=2 ** -8, atol=5e-5)
