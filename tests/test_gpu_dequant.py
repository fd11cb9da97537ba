"""The matrix-core dequantizer (csrc/tq_dequant.hip): bit-plane rows and decode-layout caches
against round(round(c[codes] R) norm) formed in float64 from the same codes.

Tolerance, per element: 2^-24 of each of the d + 1 partial sums of magnitude at most
|c| sqrt(d) (R's rows are unit vectors), times the norm, and for 16-bit results the two
roundings, half an ulp each, either of which the sum's error can move by one ulp."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"
EPS = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def check(out, codes, norms, cen, R, dt):
    d = R.shape[0]
    rd = (lambda t: t.double()) if dt == torch.float32 else (lambda t: t.to(dt).double())
    s = rd(cen)[codes.long()] @ rd(R)
    ref = s * norms.double()[..., None]
    tol = (2 * EPS[dt] + EPS[dt] ** 2) * ref.abs() + \
        (d + 1) * 2.0 ** -24 * float(cen.abs().max()) * d ** 0.5 * norms.double().abs()[..., None]
    if dt == torch.float16:
        tol = tol + 2.0 ** -24 * (1 + norms.double().abs()[..., None])  # subnormal results
    assert out.dtype == dt and bool(((out.double() - ref).abs() <= tol).all())


def data(d, bits, n, seed):
    from turboquant_kv import ops
    from turboquant_kv.codebook import lloyd_max_codebook, make_rotation_matrix
    g = torch.Generator(device=DEV).manual_seed(seed)
    codes = torch.randint(0, 1 << bits, (n, d), generator=g, device=DEV, dtype=torch.uint8)
    norms = torch.exp(torch.randn(n, generator=g, device=DEV) * 2)
    return (codes, ops.pack_codes(codes, bits), norms, lloyd_max_codebook(bits, d)[1].to(DEV),
            make_rotation_matrix(d, 42 + bits).to(DEV))


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 128])
def test_bitplane_rows(d, dt):
    """1-4 bits, row counts around the 32-token steps and the workgroups, and more rows than the
    launch's waves take in one step."""
    from turboquant_kv._lib import ops
    for bits in (1, 2, 3, 4):
        for n in (1, 15, 31, 33, 257, 20_001, 150_001):
            codes, packed, norms, cen, R = data(d, bits, n, n)
            out = ops().dequantize_mse_packed(packed, norms.to(dt), cen, R, bits, d)
            check(out, codes, norms.to(dt).float(), cen, R, dt)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d,vb", [(64, 2), (64, 3), (64, 4), (128, 2), (128, 3), (128, 4)])
def test_cache_and_new_tokens(d, vb, dt):
    """Histories around the 32- and 64-token steps, capacities past them, new tokens of any
    strides (and none); the new tokens arrive bit for bit."""
    from turboquant_kv import ops
    from turboquant_kv._lib import ops as tops
    B, H, g = 2, 3, torch.Generator(device=DEV).manual_seed(d + vb)
    for T, cap, s in ((0, 64, 2), (1, 64, 1), (31, 64, 0), (64, 64, 1), (65, 192, 3), (1000, 1024, 1)):
        kc, kp_rows, kn, kcen, kR = data(d, 4, B * H * T, 1)
        vc, vp_rows, vn, vcen, vR = data(d, vb, B * H * T, 2)
        kp = torch.randint(0, 256, (B, H, cap, d // 2), generator=g, device=DEV, dtype=torch.uint8)
        vp = torch.randint(0, 256, (B, H, cap // 64, 8 * vb * d), generator=g, device=DEV, dtype=torch.uint8)
        kno, vno = (torch.full((B, H, cap), float("nan"), device=DEV, dtype=dt) for _ in range(2))
        if T:
            ops.pack_decode_layout(kp_rows.view(B * H, T, -1), kp.view(B * H, cap, -1), d, 4, False, 0)
            ops.pack_decode_layout(vp_rows.view(B * H, T, -1), vp.view(B * H, cap // 64, -1), d, vb, True, 0)
            kno[:, :, :T], vno[:, :, :T] = kn.view(B, H, T).to(dt), vn.view(B, H, T).to(dt)
        k1 = torch.randn(B, s, H, d + 1, generator=g, device=DEV).to(dt)[..., :d].transpose(1, 2)
        v1 = torch.randn(B, s, H, d, generator=g, device=DEV).to(dt).transpose(1, 2)
        k, v = tops().dequantize_cache_dl(kp, kno, vp, vno, T, kcen, kR, vcen, vR, dt, *((k1, v1) if s else ()))
        assert k.shape == v.shape == (B, H, T + s, d)
        assert torch.equal(k[:, :, T:], k1) and torch.equal(v[:, :, T:], v1)
        if T:
            check(k[:, :, :T], kc.view(B, H, T, d), kno[:, :, :T].float(), kcen, kR, dt)
            check(v[:, :, :T], vc.view(B, H, T, d), vno[:, :, :T].float(), vcen, vR, dt)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d,vb", [(64, 2), (64, 3), (64, 4), (128, 2), (128, 3), (128, 4)])
def test_cache_of_many_tokens(d, vb, dt):
    """More 32-token steps than the launch has waves: each takes one after another, its next codes
    on their way."""
    from turboquant_kv import ops
    from turboquant_kv._lib import ops as tops
    B, H, T, cap = 8, 8, 2100, 2112
    g = torch.Generator(device=DEV).manual_seed(d + vb)
    kc, kp_rows, kn, kcen, kR = data(d, 4, B * H * T, 1)
    vc, vp_rows, vn, vcen, vR = data(d, vb, B * H * T, 2)
    kp = torch.zeros(B, H, cap, d // 2, device=DEV, dtype=torch.uint8)
    vp = torch.zeros(B, H, cap // 64, 8 * vb * d, device=DEV, dtype=torch.uint8)
    ops.pack_decode_layout(kp_rows.view(B * H, T, -1), kp.view(B * H, cap, -1), d, 4, False, 0)
    ops.pack_decode_layout(vp_rows.view(B * H, T, -1), vp.view(B * H, cap // 64, -1), d, vb, True, 0)
    kno, vno = (torch.full((B, H, cap), float("nan"), device=DEV, dtype=dt) for _ in range(2))
    kno[:, :, :T], vno[:, :, :T] = kn.view(B, H, T).to(dt), vn.view(B, H, T).to(dt)
    x = torch.randn(B, H, 3, d, generator=g, device=DEV).to(dt)
    k, v = tops().dequantize_cache_dl(kp, kno, vp, vno, T, kcen, kR, vcen, vR, dt, x, x * 2)
    assert torch.equal(k[:, :, T:], x) and torch.equal(v[:, :, T:], x * 2)
    check(k[:, :, :T], kc.view(B, H, T, d), kno[:, :, :T].float(), kcen, kR, dt)
    check(v[:, :, :T], vc.view(B, H, T, d), vno[:, :, :T].float(), vcen, vR, dt)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d,vb", [(64, 2), (64, 3), (128, 4)])
def test_cache_norms_wider_than_the_result(d, vb, dt):
    """fp32 norms of a cache are rounded to a 16-bit result's type before they are multiplied in:
    the rows of a cache that holds them rounded, bit for bit."""
    from turboquant_kv._lib import ops as tops
    g = torch.Generator(device=DEV).manual_seed(d + vb)
    B, H, cap, T = 2, 3, 128, 100
    kp = torch.randint(0, 256, (B, H, cap, d // 2), generator=g, device=DEV, dtype=torch.uint8)
    vp = torch.randint(0, 256, (B, H, cap // 64, 8 * vb * d), generator=g, device=DEV, dtype=torch.uint8)
    kn, vn = (torch.exp(torch.randn(B, H, cap, generator=g, device=DEV) * 2) for _ in range(2))
    (_, _, _, kcen, kR), (_, _, _, vcen, vR) = data(d, 4, 1, 1), data(d, vb, 1, 2)
    got = tops().dequantize_cache_dl(kp, kn, vp, vn, T, kcen, kR, vcen, vR, dt)
    want = tops().dequantize_cache_dl(kp, kn.to(dt), vp, vn.to(dt), T, kcen, kR, vcen, vR, dt)
    for a, b in zip(got, want):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))


def test_layer_update_keeps_gradients():
    """A layer's update returns tensors through which new tokens' gradients still flow."""
    from turboquant_kv.config import TurboQuantConfig
    from turboquant_kv.hf_integration import TurboQuantLayer
    outs = []
    for grad in (False, True):
        layer = TurboQuantLayer(TurboQuantConfig())
        g = torch.Generator(device=DEV).manual_seed(3)
        x = torch.randn(2, 2, 70, 64, generator=g, device=DEV)
        with torch.no_grad():
            layer.update(x, x)
        n = torch.randn(2, 2, 1, 64, generator=g, device=DEV).requires_grad_(grad)
        k, v = layer.update(n, n * 2)
        outs.append((k.detach(), v.detach()))
        assert k.requires_grad == grad
        if grad:
            (k.sum() + v.sum()).backward()
            assert torch.equal(n.grad, torch.full_like(n, 3.0))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
