"""CPU sanity tests for the reference op implementations (numerics contract).

These pin the semantics the HIP kernels are tested against.
"""
import math

import pytest
import torch

import helix_amd.ops as ops
import helix_amd.ops.reference as ref


def test_rms_norm_known_value():
    x = torch.full((1, 8), 2.0, dtype=torch.bfloat16)
    w = torch.ones(8, dtype=torch.bfloat16)
    out = ops.rms_norm(x, w, 0.0)
    assert torch.allclose(out.float(), torch.ones(1, 8), atol=1e-2)


def test_fused_add_rms_norm_semantics():
    x = torch.randn(4, 16, dtype=torch.bfloat16)
    r = torch.randn(4, 16, dtype=torch.bfloat16)
    w = torch.ones(16, dtype=torch.bfloat16)
    x2, r2 = x.clone(), r.clone()
    out, new_res = ops.fused_add_rms_norm(x2, r2, w, 1e-5)
    assert torch.allclose(new_res.float(), (x.float() + r.float()), atol=2e-2)
    assert torch.allclose(out.float(), ref.rms_norm(new_res, w, 1e-5).float(),
                          atol=1e-2)


def test_rope_preserves_norm():
    d = 64
    q = torch.randn(5, 4 * d, dtype=torch.bfloat16)
    k = torch.randn(5, 2 * d, dtype=torch.bfloat16)
    pos = torch.arange(5, dtype=torch.int64)
    cs = ref.make_cos_sin_cache(d, 16)
    q2, k2 = ops.rotary_embedding(pos, q.clone(), k.clone(), cs, d)
    # rotation preserves the per-head L2 norm
    for h in range(4):
        a = q.float().view(5, 4, d)[:, h].norm(dim=-1)
        b = q2.float().view(5, 4, d)[:, h].norm(dim=-1)
        assert torch.allclose(a, b, rtol=2e-2)
    # position 0 is identity
    assert torch.allclose(q2[0].float(), q[0].float(), atol=1e-2)


def test_silu_and_mul():
    x = torch.cat([torch.zeros(3, 8), torch.randn(3, 8)], dim=-1).bfloat16()
    out = ops.silu_and_mul(x)
    assert torch.allclose(out.float(), torch.zeros(3, 8))  # silu(0)=0


def test_attn_prefill_causal_first_token():
    """First token attends only to itself => out == v[0]."""
    q = torch.randn(7, 4, 64, dtype=torch.bfloat16)
    k = torch.randn(7, 2, 64, dtype=torch.bfloat16)
    v = torch.randn(7, 2, 64, dtype=torch.bfloat16)
    cu = torch.tensor([0, 7], dtype=torch.int32)
    out = ops.attn_prefill(q, k, v, cu, 7, 0.125)
    want0 = v[0].repeat_interleave(2, dim=0)
    assert torch.allclose(out[0].float(), want0.float(), atol=2e-2)


def test_paged_decode_matches_prefill_last_row():
    """Decode of the last position must equal prefill's last-row output."""
    torch.manual_seed(0)
    L, hq, hkv, d, bs = 37, 8, 4, 64, 16
    q = torch.randn(L, hq, d, dtype=torch.bfloat16)
    k = torch.randn(L, hkv, d, dtype=torch.bfloat16)
    v = torch.randn(L, hkv, d, dtype=torch.bfloat16)
    cu = torch.tensor([0, L], dtype=torch.int32)
    scale = d ** -0.5
    pre = ops.attn_prefill(q, k, v, cu, L, scale)

    nb = (L + bs - 1) // bs
    kc = torch.zeros(nb + 1, hkv, bs, d, dtype=torch.bfloat16)
    vc = torch.zeros_like(kc)
    slots = torch.arange(bs, bs + L, dtype=torch.int64)  # blocks 1..
    ops.reshape_and_cache(k, v, kc, vc, slots)
    bt = torch.arange(1, nb + 2, dtype=torch.int32).unsqueeze(0)
    out = ops.paged_attn_decode(q[-1:].reshape(1, hq, d), kc, vc, bt,
                                torch.tensor([L], dtype=torch.int32), scale)
    assert torch.allclose(out[0].float(), pre[-1].float(), atol=3e-2,
                          rtol=3e-2)


def test_sample_greedy_cpu():
    logits = torch.randn(4, 100, dtype=torch.bfloat16)
    temps = torch.zeros(4)
    seeds = torch.zeros(4, dtype=torch.int64)
    out = ops.sample_tokens(logits, temps, seeds)
    assert torch.equal(out, logits.float().argmax(-1))


def test_gemm_reference():
    x = torch.randn(5, 64, dtype=torch.bfloat16)
    w = torch.randn(7, 64, dtype=torch.bfloat16)
    out = ops.gemm_bf16(x, w)
    assert torch.allclose(out.float(), (x.float() @ w.float().t()), atol=0.5)


def test_cos_sin_cache():
    cs = ref.make_cos_sin_cache(8, 4, base=10000.0)
    assert cs.shape == (4, 8)
    assert torch.allclose(cs[0, :4], torch.ones(4))  # cos(0)
    assert torch.allclose(cs[0, 4:], torch.zeros(4))  # sin(0)
    assert math.isclose(float(cs[1, 0]), math.cos(1.0), rel_tol=1e-5)


def test_sliding_window_reference_consistency():
    """Windowed decode of the last position == windowed prefill last row."""
    torch.manual_seed(5)
    L, hq, hkv, d, bs, W = 50, 8, 4, 64, 16, 16
    q = torch.randn(L, hq, d, dtype=torch.bfloat16)
    k = torch.randn(L, hkv, d, dtype=torch.bfloat16)
    v = torch.randn(L, hkv, d, dtype=torch.bfloat16)
    cu = torch.tensor([0, L], dtype=torch.int32)
    scale = d ** -0.5
    pre = ops.attn_prefill(q, k, v, cu, L, scale, window=W)
    nb = (L + bs - 1) // bs
    kc = torch.zeros(nb + 1, hkv, bs, d, dtype=torch.bfloat16)
    vc = torch.zeros_like(kc)
    ops.reshape_and_cache(k, v, kc, vc,
                          torch.arange(bs, bs + L, dtype=torch.int64))
    bt = torch.arange(1, nb + 2, dtype=torch.int32).unsqueeze(0)
    out = ops.paged_attn_decode(q[-1:].reshape(1, hq, d), kc, vc, bt,
                                torch.tensor([L], dtype=torch.int32), scale,
                                window=W)
    assert torch.allclose(out[0].float(), pre[-1].float(), atol=3e-2,
                          rtol=3e-2)
    # and differs from full attention (the window actually applies)
    full = ops.attn_prefill(q, k, v, cu, L, scale)
    assert not torch.allclose(full[-1].float(), pre[-1].float(), atol=1e-3)


def _out(x, w):
    return torch.empty(x.shape[0], w.shape[0], dtype=x.dtype)


@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("bias", [False, True])
def test_gemm_bf16_without_inner_dimension(bias, act):
    """act(bias), decided on the host: there is nothing to load."""
    x, w = (torch.empty(n, 0, dtype=torch.bfloat16) for n in (3, 10))
    b = torch.randn(20, dtype=torch.bfloat16)[::2] if bias else None
    out = _out(x, w)
    ops._native().gemm_bf16(out, x, w, b, act)
    assert torch.equal(out, ref.gemm_bf16(x, w, b, act))


@pytest.mark.parametrize("case,says", [
    ("bias", "a bias of N"), ("bias type", "a bias of N"),
    ("type", "bf16 on one"), ("out", "out is"), ("host", "on the GPU")])
def test_gemm_bf16_refuses(case, says):
    """What the kernels would misread is refused before any launch."""
    x = torch.zeros(3, 64, dtype=torch.bfloat16)
    w = torch.zeros(10, 64, dtype=torch.bfloat16)
    out, b = _out(x, w), torch.zeros(10, dtype=torch.bfloat16)
    if case == "bias":
        b = b[:1]
    elif case == "bias type":
        b = b.float()
    elif case == "type":
        x = x.half()
    elif case == "out":
        out = out[:, :8]
    with pytest.raises(RuntimeError, match=says):
        ops._native().gemm_bf16(out, x, w, b, 0)


@pytest.mark.parametrize("rows,columns,stays", [
    (1, 8, True), (256, 4096, True), (1, 4104, False), (257, 1024, False),
    (257, 3072, True), (512, 4096, True), (513, 4096, False),
    (1024, 512, False)])
def test_norm_in_registers(rows, columns, stays):
    """Where the loop over a row was measured faster it is taken."""
    assert ops._native().norm_in_registers(rows, columns) == stays


@pytest.mark.parametrize("m,n,k,gelu,tile,stretches", [
    (2304, 3072, 1024, True, 56, 1), (2304, 1024, 1024, False, 52, 1),
    (300, 768, 3072, False, 22, 4), (8, 6144, 1024, False, 22, 1),
    (16600, 768, 3072, False, 78, 1)])
def test_gemm_bf16_plan(m, n, k, gelu, tile, stretches):
    """The tile and stretches of least estimated time, found without working
    out the times of all 75 or more: a host pays for them at every call."""
    plan = ops._native().gemm_bf16_plan(m, n, k, gelu, False)
    assert plan[:2] == (tile, stretches) and plan[3] <= 8
    assert ops._native().gemm_bf16_plan(m, n, k, gelu, True)[3] <= 32


@pytest.mark.parametrize("m,n,k,stretches", [
    (80, 1024, 8192, 8), (512, 512, 16384, 8), (33, 2048, 7168, 8),
    (100, 2048, 14336, 4), (1540, 14336, 4096, 0), (128, 14336, 4096, 0)])
def test_gemm_gated_plan(m, n, k, stretches):
    """Gate and other factor in stretches where one launch, which has none,
    leaves CUs idle."""
    assert ops._native().gemm_bf16_glu_plan(m, n, k)[1] == stretches


def test_gemm_bf16_plan_of_any_columns():
    """Columns that are no multiple of 8 have large tiles and stretches too."""
    plan = ops._native().gemm_bf16_plan
    assert plan(8192, 4092, 4096, False, False)[:2] == (88, 1)
    assert plan(8192, 3001, 2048, False, False)[0] == 48
    assert plan(100, 1020, 4096, False, False)[1] > 1


def test_gemm_bf16_cuts():
    """Behind the full rounds of large tiles, by rows or columns, where that
    takes less than one launch by more than the estimates are off."""
    cut, glu = ops._native().gemm_bf16_cut, ops._native().gemm_bf16_glu_cut
    assert cut(5537, 4096, 4096, False)[:3] == (True, 4096, 88)
    assert cut(3195, 6144, 4096, False)[:3] == (False, 4864, 88)
    assert glu(1540, 14336, 4096)[:2] == (False, 13952)
    assert glu(4101, 14336, 4096)[:2] == (True, 4096)
    for M, N, K in ((8192, 4096, 4096), (300, 4096, 4096), (8065, 2304, 768)):
        assert cut(M, N, K, False)[1] == 0
    for M, N, K in ((8192, 14336, 4096), (33, 14336, 4096), (1, 8, 64)):
        assert glu(M, N, K)[1] == 0
    for M in range(257, 9000, 613):
        rows, at, first, rest, us = cut(M, 4104, 2048, False)
        if at:
            assert 0 < at < (M if rows else 4104)
            assert at % (32 * (first // 10 if rows else first % 10)) == 0
            assert us < ops._native().gemm_bf16_plan(M, 4104, 2048, False,
                                                     False)[2]


def test_gemm_ring_loads_stay_at_the_start():
    """Descriptors are empty after the last item; a scalar offset is not part
    of their check, so it stays at 0 however many steps follow."""
    places = ops._native().gemm_ring_places
    assert places([0, 128, 64, 192], 9) == [0, 64, 64, 128, 0, 0, 0, 0, 0]
    assert places([0, 64], 40) == [0] * 40
    assert places([], 3) == [0, 0, 0]
    # begun elsewhere, an item goes round to its start
    assert places([0, 256], 6, 128) == [128, 192, 0, 64, 0, 0]
    assert places([0, 128, 0, 128], 6, 64) == [64, 0, 64, 0, 0, 0]


@pytest.mark.parametrize("case,says", [
    ("out shape", "out is packed"), ("out rows", "out is packed"),
    ("q", "q is packed"), ("cache", "caches are"), ("pages", "caches are"),
    ("lens", "a length and"), ("table", "a length and"),
    ("workspace", "a workspace of"), ("host", "on one GPU")])
def test_paged_attn_decode_refuses(case, says):
    """What would be read or written out of range is refused before any
    launch."""
    q = torch.zeros(3, 4, 64, dtype=torch.bfloat16)
    kc = torch.zeros(9, 2, 128, 64, dtype=torch.bfloat16)
    vc, out = kc.clone(), torch.empty_like(q)
    bt = torch.zeros(3, 3, dtype=torch.int32)
    lens = torch.full((3,), 300, dtype=torch.int32)
    ws = ops.decode_workspace(2 if case == "workspace" else 3, 4, 64, 384,
                              "cpu")
    if case == "out shape":
        out = out[:2]
    elif case == "out rows":
        out = torch.empty(3, 4, 128, dtype=torch.bfloat16)[..., :64]
    elif case == "q":
        q = torch.zeros(3, 64, 4, dtype=torch.bfloat16).transpose(1, 2)
    elif case == "cache":
        vc = vc.half()
    elif case == "pages":
        kc = kc[:, :, ::2]
    elif case == "lens":
        lens = lens[:2]
    elif case == "table":
        bt = bt[:2]
    with pytest.raises(RuntimeError, match=says):
        ops._native().paged_attn_decode(out, q, kc, vc, bt, lens, 0.125,
                                        *ws, 384, 0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_fused_add_rms_norm_of_batches(dtype):
    """[B, T, H] is a batch of rows, not a product's stretches."""
    x, r = torch.randn(2, 3, 5, 16, dtype=dtype)
    w = torch.randn(16, dtype=dtype)
    want = ref.fused_add_rms_norm(x, r, w, 1e-5)
    got = ops.fused_add_rms_norm(x.clone(), r.clone(), w, 1e-5)
    for a, b in zip(got, want):
        assert a.shape == (3, 5, 16) and torch.equal(a, b)


def test_linear_with_a_vector():
    """A weight of one dimension, as torch's linear takes it."""
    x, w = torch.randn(5, 16), torch.randn(16)
    for z in (x, x[0]):
        assert torch.equal(ops.linear(z, w),
                           torch.nn.functional.linear(z, w))


@pytest.mark.parametrize("M,N,K,pay", [
    (128, 4096, 14336, True), (130, 4096, 14336, True),
    (512, 4096, 14336, True), (1540, 4096, 14336, True),
    (2049, 4096, 14336, False), (640, 8192, 28672, True),
    (2048, 8192, 28672, False), (200, 1024, 4096, True),
    (2048, 1024, 4096, False), (1024, 4096, 4096, False),
    (200, 8200, 32768, False), (130, 8, 64, False), (65, 2048, 2048, True),
    (129, 4096, 4096, True), (200, 4096, 4096, True), (400, 4096, 4096, False),
    (300, 512, 1280, False), (128, 16, (1 << 21) + 256, True),
    (129, 16, (1 << 21) + 256, False)])
def test_sums_pay(M, N, K, pay):
    """Stretches where they are the faster form with their reader: at the ends
    of the range, where tiles alone fill the chip, where there is little to
    do, beyond the offsets of tiles."""
    assert ops._sums_pay(M, N, K) == pay


@pytest.mark.parametrize("M,N,K,streamed", [
    (16, 8192, 28672, True), (17, 8192, 28672, False),
    (48, 2048, 2048, True), (49, 2048, 2048, False), (64, 4096, 768, True),
    (65, 4096, 768, False), (17, 3072, 1536, False), (64, 1024, 16384, True),
    (64, 1024, 8192, False), (24, 7168, 8192, True), (33, 7168, 8192, False),
    (64, 8192, 8192, True)])
def test_sums_streamed(M, N, K, streamed):
    assert ops._sums_streamed(M, N, K) == streamed


def test_few_rows_where_they_pay():
    """The lines between the gated products of few rows and the library's."""
    glu = ops._glu_fits
    assert glu(1, 28672, 4096) and glu(16, 12288, 4096) and glu(64, 64, 1024)
    assert glu(17, 28672, 4096) and glu(64, 26624, 2048)
    assert not (glu(1, 8192, 4096) or glu(17, 26560, 4096) or
                glu(32, 28672, 5120) or glu(64, 57344, 8192))


@pytest.mark.parametrize("M,N,K,pay", [
    (128, 28672, 4096, False), (129, 28672, 4096, True),
    (48, 768, 4096, False), (64, 768, 4096, True), (64, 768, 16384, False),
    (256, 2048, 2048, False), (257, 2048, 2048, True),
    (128, 2560, 2048, True), (127, 2560, 2048, False), (24, 1536, 2048, True),
    (512, 1024, 1280, False), (577, 1024, 1280, True), (128, 512, 3072, True),
    (129, 512, 3072, False), (192, 768, 768, False), (193, 768, 768, True),
    (100, 256, 768, True), (100, 256, 1024, False), (32, 1024, 1024, False),
    (33, 1280, 1024, True), (100, 512, 512, True), (300, 6144, 4096, True),
    (127, 8192, 8192, False), (128, 8192, 8192, True), (32, 7168, 8192, False),
    (48, 7168, 8192, True), (32, 8192, 28672, True)])
def test_tiles_pay(M, N, K, pay):
    """Where tiles were measured slower than what products took before them,
    that is taken."""
    assert ops._tiles_pay(M, N, K) == pay


@pytest.mark.parametrize("M,N,K,way", [
    (16, 128256, 4096, "stream"), (16, 65537, 3584, "library"),
    (16, 65536, 3584, "stream"), (24, 28672, 4096, "tiles"),
    (24, 32776, 4096, "stream"), (32, 128256, 2048, "stream"),
    (33, 128256, 4096, "tiles"), (48, 24576, 2048, "stream"),
    (49, 24576, 2048, "library"), (48, 24568, 2048, "library"),
    (128, 24576, 8192, "tiles"), (32, 28672, 8192, "library"),
    (128, 24568, 4096, "library"), (129, 24568, 4096, "tiles"),
    (61, 37888, 3584, "library"),
    # vocabularies
    (8, 65537, 768, "stream"), (9, 65537, 768, "library"),
    (8, 65537, 5120, "library"), (8, 65537, 512, "library"),
    (17, 128256, 3584, "tiles"), (32, 86016, 768, "tiles"),
    (32, 85888, 768, "stream"), (32, 81920, 4096, "stream"),
    (32, 128256, 4096, "tiles"), (33, 128256, 2560, "library"),
    (128, 100352, 1536, "tiles"), (64, 128256, 2048, "stream"),
    (65, 128256, 2048, "library"), (17, 128256, 5120, "library")])
def test_wide_products(M, N, K, way):
    """Streamed, by tiles or by the library, on either side of the lines."""
    tiles = M > 16 and (ops._tiles_pay(M, N, K)
                        or ops._tiles_apart_pay(M, N, K))
    assert way == ("tiles" if tiles else
                   "stream" if ops._streams_pay(M, N, K) else "library")


@pytest.mark.parametrize("case,says", [
    ("type", "rows are bf16"), ("out", "rows are bf16"),
    ("keys", "a boundary more"), ("host", "on one GPU")])
def test_attn_prefill_refuses(case, says):
    """What would be misread, or read by the host's addresses, is refused
    before any launch."""
    q, k, v, out = (torch.zeros(9, 2, 64, dtype=torch.bfloat16)
                    for _ in range(4))
    cu = torch.tensor([0, 4, 9], dtype=torch.int32)
    cu_k = cu
    if case == "type":
        k = k.half()
    elif case == "out":
        out = out.float()
    elif case == "keys":
        cu_k = cu[:2]
    with pytest.raises(RuntimeError, match=says):
        ops._native().attn_prefill(out, q, k, v, cu, cu_k, 5, 0.125, True, 0)


@pytest.mark.parametrize("gone", range(12))
def test_blocks_without_a_bias_go_step_by_step(gone):
    """A parameter that is None is a form that the calls decline, not an
    argument that they refuse."""
    x, cu = torch.zeros(4, 64, dtype=torch.bfloat16), torch.tensor([0, 4]).int()
    params = [None if i == gone else x for i in range(12)]
    native = ops._native()
    assert native.text_block(x, cu, 4, 1, 1.0, 1e-6, params) is None
    assert native.image_block(x, None, None, None, x, cu, 4, 1, 1.0, 1e-6,
                              params[:10], True) == []
    assert native.gemm_rows_many(x, [x, x], [x, None]) == []
