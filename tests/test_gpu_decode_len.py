"""Decode over the first `length` tokens of a decode-layout cache, the length an argument:
against the same call with a tensor of lengths (its splits are planned for the capacity, so
the fp32 sums come in another order)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("d,vb,B,hkv,G", [(64, 2, 1, 8, 4), (128, 3, 3, 2, 1), (64, 4, 2, 1, 5), (128, 2, 1, 1, 8)])
def test_length_argument_vs_length_tensor(d, vb, B, hkv, G):
    from turboquant_kv import ops
    from turboquant_kv.codebook import lloyd_max_codebook, make_rotation_matrix
    tc = 2048
    g = torch.Generator(device=DEV).manual_seed(d + vb)
    kp = torch.randint(0, 256, (B, hkv, tc, d // 2), dtype=torch.uint8, generator=g, device=DEV)
    vt = torch.randint(0, 256, (B, hkv, tc // 64, 8 * vb * d), dtype=torch.uint8, generator=g, device=DEV)
    kn, vn = (torch.rand(B, hkv, tc, generator=g, device=DEV) * 4 + 1 for _ in range(2))
    kc, vc = (lloyd_max_codebook(b, d)[1].to(DEV) for b in (4, vb))
    R = make_rotation_matrix(d, seed=1).to(DEV)
    q = torch.randn(B, hkv * G, d, generator=g, device=DEV)
    for T in (0, 1, 63, 64, 65, 700, 1025, tc):
        args = (kc, vc, R, R, 0.125)
        want = ops.decode_attention_dl(q, kp, kn, vt, vn, torch.full((B,), T, dtype=torch.int32, device=DEV), *args)
        got = ops.decode_attention_dl_len(q, kp, kn, vt, vn, T, *args)
        # fp32-accurate both: the split sums' order only (128 partial sums: 2^-24 * 128 < 4e-5)
        assert got.shape == want.shape and got.dtype == want.dtype
        assert (got - want).abs().max() <= 4e-5 * want.abs().max()
    for bad in (-1, tc + 1):
        with pytest.raises(RuntimeError, match="length"):
            ops.decode_attention_dl_len(q, kp, kn, vt, vn, bad, kc, vc, R, R, 0.125)
