"""GPU: the decoder-layer kernels (include/flexengine_amd_model.h) against
plain PyTorch restatements of the ops they fuse (fp16 element-wise semantics)
and an fp32 matrix product for the skinny GEMM, including ragged sizes."""
from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from flexengine_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def randn(*shape, seed=0, scale=1.0):
    return (torch.randn(shape, generator=gen(seed), device=DEV) * scale).half()


def torch_rmsnorm(x, w, eps, residual=None):
    r = x if residual is None else x + residual  # fp16 add
    f = r.float()
    return w * (f * torch.rsqrt(f.square().mean(-1, keepdim=True) + eps)).half(), r


def ulps(a, b):
    """max difference in fp16 units in the last place of b."""
    d = (a.float() - b.float()).abs()
    ulp = torch.where(b.float().abs() < 6.1e-5, torch.full_like(d, 6e-8),
                      2.0 ** (torch.floor(torch.log2(b.float().abs().clamp_min(6.1e-5))) - 10))
    return (d / ulp).max().item()


@pytest.mark.parametrize("rows,hidden", [(1, 1536), (5, 1536), (64, 896), (3, 8192)])
def test_rmsnorm_matches_torch(rows, hidden):
    """The sum of squares adds in another order than PyTorch's, so fp16(r * rsqrt(..))
    can round one ulp apart for a rare element, which the weight multiply scales by |w|
    (here N(0, 1)): at most 2 ulps, nearly all elements bit-identical."""
    x, res, w = randn(rows, hidden, seed=1), randn(rows, hidden, seed=2), randn(hidden, seed=3)
    out, _ = ops.rmsnorm(x, w, 1e-6)
    want, _ = torch_rmsnorm(x, w, 1e-6)
    assert ulps(out, want) <= 2 and (out == want).float().mean() > 0.999
    r = res.clone()
    out, r2 = ops.rmsnorm(x, w, 1e-6, residual=r)
    want, want_r = torch_rmsnorm(x, w, 1e-6, residual=res)
    assert r2 is r and torch.equal(r, want_r)          # residual add is bit-exact
    assert ulps(out, want) <= 2 and (out == want).float().mean() > 0.999


def test_rmsnorm_reads_skinny_partials():
    x, w_lin, w = randn(7, 256, seed=4), randn(1536, 256, seed=5, scale=0.1), randn(1536, seed=6)
    res = randn(7, 1536, seed=7)
    part = ops.gemm_skinny(x, w_lin)
    o16 = part.sum(0).half()
    r = res.clone()
    out, _ = ops.rmsnorm(part, w, 1e-6, residual=r)
    want, want_r = torch_rmsnorm(o16, w, 1e-6, residual=res)
    assert ulps(r, want_r) <= 1 and ulps(out, want) <= 2


def emulated_rope(x16, positions, inv_freq):
    """RoPE of fp16 rows x16 [rows, H, D] with the kernel's rounding sequence, on the
    CPU: angle = fp32(pos * inv_freq); c, s = fp16 of the correctly rounded cos/sin
    (float64); each product and sum rounded to fp16."""
    x = x16.cpu().float()
    half = x.shape[-1] // 2
    ang = positions.cpu().float()[:, None] * inv_freq.cpu()[None, :]        # fp32 product
    c = ang.double().cos().half().float()[:, None, :]
    s = ang.double().sin().half().float()[:, None, :]
    a, b = x[..., :half], x[..., half:]
    r16 = lambda t: t.half().float()
    o1 = r16(r16(a * c) + r16(-b * s))
    o2 = r16(r16(b * c) + r16(a * s))
    bound = 2.0 ** (torch.floor(torch.log2((a.abs() + b.abs()).clamp_min(2 ** -14))) - 9)
    return torch.cat([o1, o2], -1), torch.cat([bound, bound], -1)


@pytest.mark.parametrize("rows,hq,hkv,d", [(1, 12, 2, 128), (9, 14, 2, 64), (33, 4, 4, 128)])
def test_rope_qkv_matches_emulated_rounding(rows, hq, hkv, d):
    qkv = randn(rows, (hq + 2 * hkv) * d, seed=8)
    positions = torch.randint(0, 40000, (rows,), generator=gen(9), device=DEV)
    positions[0] = 0
    inv_freq = 1.0 / 1e6 ** (torch.arange(0, d, 2, device=DEV, dtype=torch.float32) / d)
    q, k, v = ops.rope_qkv(qkv, positions, inv_freq, hq, hkv, d)
    for got, src in ((q, qkv[:, :hq * d].view(rows, hq, d)),
                     (k, qkv[:, hq * d:(hq + hkv) * d].view(rows, hkv, d))):
        want, bound = emulated_rope(src, positions, inv_freq)
        err = (got.cpu().float() - want).abs()
        # exact but for a cos/sin whose fp16 rounding flips: 2 ulps of |x1| + |x2|
        assert (err <= bound).all()
        assert (err == 0).float().mean() > 0.99
    assert torch.equal(v, qkv[:, (hq + hkv) * d:].reshape(rows, hkv, d))
    # position 0 is the identity
    assert torch.equal(q[0], qkv[0, :hq * d].view(hq, d))


def test_rope_qkv_from_partials_adds_bias():
    rows, hq, hkv, d, hidden = 4, 12, 2, 128, 512
    h, w = randn(rows, hidden, seed=10), randn((hq + 2 * hkv) * d, hidden, seed=11, scale=0.05)
    bias = randn((hq + 2 * hkv) * d, seed=12)
    positions = torch.tensor([0, 1, 511, 4095], device=DEV)
    inv_freq = 1.0 / 1e6 ** (torch.arange(0, d, 2, device=DEV, dtype=torch.float32) / d)
    q, k, v = ops.rope_qkv(ops.gemm_skinny(h, w), positions, inv_freq, hq, hkv, d, bias=bias)
    qkv = (h.float() @ w.float().t() + bias.float()).half()   # one rounding, like a library GEMM
    q2, k2, v2 = ops.rope_qkv(qkv, positions, inv_freq, hq, hkv, d)
    # the fp32 sums differ only in order: inputs equal or one fp16 ulp apart
    for a, b in ((q, q2), (k, k2), (v, v2)):
        assert (a.float() - b.float()).abs().max() <= 2 ** -8 * (1 + b.float().abs().max())


@pytest.mark.parametrize("rows,inter", [(1, 8960), (16, 4864), (40, 128)])
def test_silu_mul_matches_torch(rows, inter):
    gu = randn(rows, 2 * inter, seed=13, scale=3.0)
    out = ops.silu_mul(gu)
    want = F.silu(gu[:, :inter]) * gu[:, inter:]
    assert ulps(out, want) <= 1


def _off(t, elems):
    """A copy of rows t at an offset of `elems` from an aligned start, rows `elems` longer."""
    rows, cols = t.shape
    buf = torch.zeros((rows, cols + elems), dtype=t.dtype, device=t.device)
    buf[:, elems:] = t
    return buf[:, elems:]


@pytest.mark.parametrize("rows,hq,hkv,d", [(1, 1, 1, 16), (70, 3, 1, 48), (130, 14, 2, 64),
                                           (65, 12, 2, 128), (3, 2, 1, 512), (2, 2, 1, 24)])
def test_rope_row_and_element_forms_agree(rows, hq, hkv, d):
    """The workgroup-per-row form against the element form (taken for the same rows one
    element off alignment): the same operations in the same order, so bit-identical."""
    qkv = randn(rows, (hq + 2 * hkv) * d, seed=21)
    positions = torch.randint(0, 40000, (rows,), generator=gen(22), device=DEV)
    inv_freq = 1.0 / 1e6 ** (torch.arange(0, d, 2, device=DEV, dtype=torch.float32) / d)
    want = ops.rope_qkv(_off(qkv, 1), positions, inv_freq, hq, hkv, d)
    for src in (qkv, _off(qkv, 8)):
        for got, w in zip(ops.rope_qkv(src, positions, inv_freq, hq, hkv, d), want):
            assert torch.equal(got, w)


@pytest.mark.parametrize("rows,inter", [(1, 8), (3, 2040), (67, 2056), (5, 20), (70000, 8)])
def test_silu_vector_and_element_forms_agree(rows, inter):
    """Bit-identical, infinities and NaN included (inter 20 has the element form only)."""
    gu = randn(rows, 2 * inter, seed=23, scale=3.0)
    gu[0, 0], gu[0, 1], gu[0, inter + 2], gu[0, 3] = float("inf"), float("-inf"), float("nan"), 88.0
    want = ops.silu_mul(_off(gu, 1))
    for src in (gu, _off(gu, 8)):
        assert torch.equal(ops.silu_mul(src).view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("rows,hq,hkv,d", [(95, 64, 8, 128), (96, 64, 8, 128), (97, 33, 2, 64),
                                           (96, 1, 1, 512)])
def test_rope_forms_agree_around_the_rule(rows, hq, hkv, d):
    """Rows of more chunks than a workgroup has threads take the row form from 96 rows."""
    qkv = randn(rows, (hq + 2 * hkv) * d, seed=25)
    positions = torch.randint(0, 40000, (rows,), generator=gen(26), device=DEV)
    inv_freq = 1.0 / 1e6 ** (torch.arange(0, d, 2, device=DEV, dtype=torch.float32) / d)
    want = ops.rope_qkv(_off(qkv, 1), positions, inv_freq, hq, hkv, d)
    for got, w in zip(ops.rope_qkv(qkv, positions, inv_freq, hq, hkv, d), want):
        assert torch.equal(got, w)


def test_rope_of_more_rows_than_a_launch_has_workgroups():
    """2^25 + 3 rows: a workgroup a row would be 2^32 threads and more, which no launch takes."""
    rows, d = (1 << 25) + 3, 16
    qkv = torch.empty(rows, 3 * d, dtype=torch.float16, device=DEV).normal_(generator=gen(27))
    positions = torch.arange(rows, device=DEV) % 40000
    inv_freq = 1.0 / 1e6 ** (torch.arange(0, d, 2, device=DEV, dtype=torch.float32) / d)
    got = ops.rope_qkv(qkv, positions, inv_freq, 1, 1, d)
    edge = torch.tensor([0, 1, (1 << 20) - 1, 1 << 20, (1 << 20) + 1, 1 << 24, rows - 4, rows - 1],
                        device=DEV)
    want = ops.rope_qkv(_off(qkv[edge], 1), positions[edge], inv_freq, 1, 1, d)
    for x, w in zip(got, want):
        assert torch.equal(x[edge], w)


@pytest.mark.parametrize("rows,inter", [(128, 1024), (127, 1024), (200, 1016), (64, 2056), (9, 20480)])
def test_silu_forms_agree_around_the_rule(rows, inter):
    """The vector form from 2^17 outputs in rows of 1024 and more, ragged last workgroups."""
    gu = randn(rows, 2 * inter, seed=28, scale=3.0)
    gu[0, 0], gu[0, 1], gu[0, inter + 2], gu[0, 3] = float("inf"), float("-inf"), float("nan"), 88.0
    want = ops.silu_mul(_off(gu, 1))
    assert torch.equal(ops.silu_mul(gu).view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("m,n,k", [(1, 2048, 1536), (3, 1536, 8960), (8, 17920, 1536),
                                   (16, 1000, 96), (17, 300, 1536), (32, 151936, 1536)])
def test_gemm_skinny_matches_fp32_product(m, n, k):
    x, w = randn(m, k, seed=14), randn(n, k, seed=15, scale=0.05)
    part = ops.gemm_skinny(x, w)
    assert part.shape[1:] == (m, n)
    want = x.float() @ w.float().t()
    got = part.sum(0)
    err = (got - want).abs().max().item()
    assert err <= 1e-4 * (1 + want.abs().max().item()), err


def test_gemm_skinny_rejects_unsupported_shapes():
    from flexengine_amd._lib import FlexEngineAMDError
    with pytest.raises(FlexEngineAMDError):
        ops.gemm_skinny(randn(33, 64), randn(16, 64))
    with pytest.raises(FlexEngineAMDError):
        ops.gemm_skinny(randn(2, 40), randn(16, 40))
