"""A layer's projections of a few rows, with norm, rotation and residual in their
launches (layer_rows.hip), against the same in 64 bits. Sums are fp32 over K, so
what a result differs by is its rounding to bf16 (2^-8 of its size)."""
import pytest
import torch

import helix_amd.ops as ops

pytestmark = pytest.mark.gpu

DEV = "cuda"
EPS = 1e-5


def _near(got, want):
    got, want = got.double(), want.double()
    scale = want.square().mean().sqrt()
    assert ((got - want).norm() / want.norm()).item() < 2.5e-3
    assert ((got - want).abs() <= 2 ** -8 * want.abs() + 1e-3 * scale).all()


def _rows(m, k, parts=0):
    g = torch.Generator(device=DEV).manual_seed(m * 7919 + k + parts)
    r = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    x = r(m, k).bfloat16()
    sq = r(m, parts).square() * (k / parts) if parts else None
    inv = torch.rsqrt(sq.double().sum(1, keepdim=True) / k + EPS) if parts \
        else 1.0
    return r, x, sq, inv


# one chunk, fewer than waves, shares that differ, and the presets' depths
@pytest.mark.parametrize("m,n,k", [
    (1, 64, 256), (4, 128, 512), (5, 64, 768), (8, 256, 1024), (9, 192, 1280),
    (16, 4096, 4096), (1, 4096, 14336), (15, 3584, 18944), (2, 8192, 8192)])
def test_join(m, n, k):
    r, x, _, _ = _rows(m, k)
    w, norm = (r(n, k) * 0.02).bfloat16(), (1 + 0.1 * r(n)).bfloat16()
    res = r(m, n).bfloat16()
    want = res.double() + x.double() @ w.double().t()
    out, sq = ops._native().layer_rows_join(x, w, res, norm)
    _near(res, want)
    _near(out, want * norm.double())
    torch.testing.assert_close(sq.double().sum(1), want.square().sum(1),
                               rtol=1e-4, atol=0)


@pytest.mark.parametrize("m,n,k,parts", [
    (1, 32, 256, 4), (3, 96, 512, 0), (4, 14336, 4096, 256), (7, 64, 1024, 64),
    (8, 512, 3584, 224), (13, 256, 8192, 512), (16, 14336, 4096, 256)])
def test_glu(m, n, k, parts):
    r, x, sq, inv = _rows(m, k, parts)
    w = (r(2 * n, k) * 0.02).bfloat16()
    g, u = ((x.double() @ w.double().t()) * inv).chunk(2, 1)
    _near(ops._native().layer_rows_glu(x, w, sq, EPS),
          torch.nn.functional.silu(g) * u)


@pytest.mark.parametrize("m,k,parts,hq,hkv,d,bs,fp8,bias,want_kv", [
    (1, 4096, 256, 32, 8, 128, 16, False, False, False),
    (4, 256, 4, 4, 2, 64, 16, True, True, True),
    (5, 512, 0, 6, 2, 96, 24, False, True, True),
    (8, 3584, 224, 28, 4, 128, 16, True, True, False),
    (16, 1024, 64, 8, 8, 32, 8, False, False, True),
    (17, 512, 0, 4, 2, 64, 16, False, True, True),
    (32, 4096, 0, 32, 8, 128, 16, True, False, False)])
def test_qkv(m, k, parts, hq, hkv, d, bs, fp8, bias, want_kv):
    r, x, sq, inv = _rows(m, k, parts)
    n = (hq + 2 * hkv) * d
    w = (r(n, k) * 0.02).bfloat16()
    b = r(n).bfloat16() if bias else None
    cs = ops.make_cos_sin_cache(d, 1024, 10000.0).to(DEV)
    pos = torch.arange(m, device=DEV) * 29 + 3          # up to 902
    slots = torch.randperm(4 * m * bs, device=DEV)[:m]
    slots[m // 2] = -1 if m > 1 else slots[m // 2]      # padding: not written
    kc, vc = (torch.zeros(4 * m, hkv, bs, d, device=DEV, dtype=torch.uint8 if
                          fp8 else torch.bfloat16) for _ in range(2))
    q, ko, vo = ops.rows_qkv(
        pos, x if sq is None else ops.Unscaled(x, sq, EPS), w, b, cs, hq, hkv,
        d, (kc, vc), slots, want_kv)
    y = (x.double() @ w.double().t()) * inv
    if bias:
        y += b.double()
    y = y.view(m, -1, d)
    c, s = cs[pos].double()[:, None].chunk(2, -1)
    u, v = y.chunk(2, -1)
    t = torch.cat([u * c - v * s, v * c + u * s], -1)
    _near(q, t[:, :hq])
    assert (ko is None) == (vo is None) == (not want_kv)
    if want_kv:
        _near(ko, t[:, hq:hq + hkv])
        _near(vo, y[:, hq + hkv:])
    there = slots >= 0
    for cache, want in ((kc, t[:, hq:hq + hkv]), (vc, y[:, hq + hkv:])):
        got = cache.view(torch.float8_e4m3fn).float() if fp8 else cache
        at = slots[there]
        got_rows = got[at // bs, :, at % bs]
        if fp8:                       # rounded once more, to 3 bits
            assert ((got_rows.double() - want[there]).abs()
                    <= 2 ** -4 * want[there].abs() + 2 ** -9).all()
        else:
            _near(got_rows, want[there])
        got[at // bs, :, at % bs] = 0
        assert not got.any()


@pytest.mark.parametrize("m,k,hq,hkv,d,fp8", [
    (1, 512, 4, 2, 64, False), (4, 4096, 32, 8, 128, False),
    (8, 1536, 4, 4, 32, True), (13, 512, 6, 2, 96, False),
    (17, 1024, 4, 2, 64, True), (32, 4096, 32, 8, 128, False)])
def test_qkv_bytes(m, k, hq, hkv, d, fp8):
    r, x, _, _ = _rows(m, k)
    n = (hq + 2 * hkv) * d
    w8, ws = ops.quantize_fp8((r(n, k) * 0.02).bfloat16())
    x8 = ops.Quantized(*ops.quantize_fp8(x))
    cs = ops.make_cos_sin_cache(d, 512, 10000.0).to(DEV)
    pos = torch.arange(m, device=DEV) * 15
    kc, vc = (torch.zeros(m, hkv, 16, d, device=DEV, dtype=torch.uint8 if fp8
                          else torch.bfloat16) for _ in range(2))
    slots = torch.randperm(m * 16, device=DEV)[:m]
    if m > 1:
        slots[m // 2] = -1                              # padding: not written
    q, ko, vo = ops.rows_qkv(pos, x8, w8, None, cs, hq, hkv, d, (kc, vc),
                             slots, True, ws)
    back = lambda b, s: (b.view(torch.float8_e4m3fn).double()  # noqa: E731
                         * s.double()[:, None])
    y = (back(*x8) @ back(w8, ws).t()).view(m, -1, d)
    c, s = cs[pos].double()[:, None].chunk(2, -1)
    u, v = y.chunk(2, -1)
    t = torch.cat([u * c - v * s, v * c + u * s], -1)
    _near(q, t[:, :hq])
    _near(ko, t[:, hq:hq + hkv])
    _near(vo, y[:, hq + hkv:])
    there = slots >= 0
    at = slots[there]
    for cache, rows, want in ((kc, ko, t[:, hq:hq + hkv]),
                              (vc, vo, y[:, hq + hkv:])):
        got = cache[at // 16, :, at % 16]
        if fp8:               # of sums before they were rounded to bf16: 3 bits
            want = want[there]
            assert ((got.view(torch.float8_e4m3fn).double() - want).abs()
                    <= 2 ** -4 * want.abs() + 2 ** -9).all()
        else:
            assert torch.equal(got, rows[there])
        cache[at // 16, :, at % 16] = 0
        assert not cache.any()


def test_refuses():
    C = ops._native()
    x = torch.zeros(17, 256, device=DEV, dtype=torch.bfloat16)
    w = torch.zeros(64, 256, device=DEV, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError):
        C.layer_rows_glu(x, w, None, EPS)              # too many rows
    with pytest.raises(RuntimeError):
        C.layer_rows_glu(x[:2, :128].contiguous(), w, None, EPS)
    with pytest.raises(RuntimeError):
        C.layer_rows_join(x[:2], w, x[:2, :32].contiguous(), w[0])
    with pytest.raises(RuntimeError):
        C.layer_rows_glu(x[:2], w, torch.zeros(2, 6, device=DEV), EPS)
