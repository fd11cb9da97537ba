"""The decode kernel's own merge of the exact current token against the decode op followed by
the merge op: the same arithmetic in the same order, so equal bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


# one split / several / two streams per workgroup (512 streams of one split); both head
# dims; more than four query heads per KV head; lengths 0, one tile's edge, the capacity
@pytest.mark.parametrize("d,vb,B,hkv,G,tc,norm", [
    (64, 2, 3, 2, 4, 256, torch.float32), (64, 3, 2, 1, 5, 4096, torch.bfloat16),
    (64, 4, 33, 16, 3, 128, torch.bfloat16), (128, 3, 3, 2, 1, 256, torch.float32),
    (128, 2, 2, 1, 8, 4096, torch.float16), (64, 3, 171, 3, 2, 512, torch.float32)])
@pytest.mark.parametrize("dt,kv_dt", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32),
                                      (torch.float32, torch.float16)])
def test_merged_equals_decode_then_merge(d, vb, B, hkv, G, tc, norm, dt, kv_dt):
    from turboquant_kv._lib import ops
    from turboquant_kv.codebook import lloyd_max_codebook, make_rotation_matrix
    g = torch.Generator(device=DEV).manual_seed(d + vb + B)
    kp = torch.randint(0, 256, (B, hkv, tc, d // 2), dtype=torch.uint8, generator=g, device=DEV)
    vt = torch.randint(0, 256, (B, hkv, tc // 64, 8 * vb * d), dtype=torch.uint8, generator=g, device=DEV)
    kn, vn = ((torch.rand(B, hkv, tc, generator=g, device=DEV) * 4 + 1).to(norm) for _ in range(2))
    kc, vc = (lloyd_max_codebook(b, d)[1].to(DEV) for b in (4, vb))
    R = make_rotation_matrix(d, seed=1).to(DEV)
    q = torch.randn(B, hkv * G, d, generator=g, device=DEV).to(dt)
    k1, v1 = (torch.randn(B, hkv, d, generator=g, device=DEV).to(kv_dt) for _ in range(2))
    lens = torch.randint(0, tc + 1, (B,), dtype=torch.int32, generator=g, device=DEV)
    lens[0], lens[-1] = 0, tc
    for starts in (None, (lens // 3).to(torch.int32)):
        args = (q, kp, kn, vt, vn, lens, kc, vc, R, R, 0.125, starts)
        o, lse = ops().decode_attention_dl_lse(*args)
        want = ops().decode_merge_token(o, lse, q, k1, v1, 0.125)
        got = ops().decode_attention_dl_merged(*args, k1, v1)
        assert got.dtype == want.dtype and torch.equal(got, want)
        assert torch.equal(got[0], v1[0].repeat_interleave(G, 0).to(dt))  # no history: its own value


@pytest.mark.parametrize("d", [64, 128])
def test_merge_rounds_the_new_value_then_the_sum(d):
    """o e^(lse - m) + v e^(s - m) is rounded as one fma over the rounded second product: with s = 20
    above lse the weights are e^-20 (read back from o = 1, v = 0) and 1, their sum 1."""
    from turboquant_kv._lib import ops
    g = torch.Generator(device=DEV).manual_seed(d)
    q, k = torch.zeros(2, 8, d, device=DEV), torch.zeros(2, 2, d, device=DEV)
    q[..., 0], k[..., 0] = 4.0, 5.0
    lse = torch.zeros(2, 8, device=DEV)
    w = ops().decode_merge_token(torch.ones_like(q), lse, q, k, torch.zeros_like(k), 1.0)
    assert torch.equal(w, w[0, 0, 0].expand_as(w)) and abs(float(w[0, 0, 0]) / 2.0611536e-09 - 1) < 1e-6
    o = torch.randn(2, 8, d, generator=g, device=DEV) * 4e8
    v = torch.randn(2, 2, d, generator=g, device=DEV)
    got = ops().decode_merge_token(o, lse, q, k, v, 1.0)
    want = (o.double() * w.double() + v.repeat_interleave(4, 1).double()).float()  # 48-bit product: exact
    assert torch.equal(got, want)
