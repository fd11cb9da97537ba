"""bf16 / fp16 keys and values quantized straight into decode-layout caches and paged pools
(csrc/tq_append.hip) against the separate quantize, layout and store ops: the same bytes,
other tokens' bits untouched."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


def tables(d, vb):
    from turboquant_kv.codebook import lloyd_max_codebook, make_rotation_matrix
    t = lambda x: x.to(DEV)  # noqa: E731
    return (t(make_rotation_matrix(d, 42)), t(lloyd_max_codebook(4, d)[0]),
            t(make_rotation_matrix(d, 43)), t(lloyd_max_codebook(vb, d)[0]))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d,vb", [(64, 2), (64, 3), (64, 4), (128, 2), (128, 3), (128, 4)])
def test_cache_append(d, vb, dt):
    """Positions and lengths around the 16-token sub-blocks and 64-token tiles, one token per
    stream included; contiguous, transposed and unaligned rows; norms in both types."""
    g = torch.Generator(device=DEV).manual_seed(10 * d + vb)
    for pos, n in ((0, 1), (63, 1), (38, 1), (0, 16), (5, 3), (15, 2), (16, 48), (7, 130), (0, 256), (61, 65)):
        for form in ("contiguous", "transposed", "odd"):
            append_equals_separate_ops(3, 7, 256, pos, n, d, vb, dt, form, g)


@pytest.mark.parametrize("d,vb", [(64, 2), (64, 3), (64, 4), (128, 2), (128, 3), (128, 4)])
def test_cache_append_large(d, vb):
    """More 16-token sub-blocks than the launch has waves, from an odd position; one token of more
    streams than its waves take at once."""
    g = torch.Generator(device=DEV).manual_seed(10 * d + vb)
    append_equals_separate_ops(8, 8, 1088, 37, 1000, d, vb, torch.bfloat16, "transposed", g)
    append_equals_separate_ops(5000, 7, 64, 37, 1, d, vb, torch.bfloat16, "contiguous", g)


@pytest.mark.parametrize("d,vb", [(64, 3), (128, 2), (128, 3), (128, 4)])
def test_cache_append_rotation_at_any_address(d, vb):
    """Rotations that are not 16-byte aligned: one token a stream and several."""
    g = torch.Generator(device=DEV).manual_seed(d + vb)
    for pos, n in ((38, 1), (5, 40)):
        append_equals_separate_ops(3, 7, 256, pos, n, d, vb, torch.bfloat16, "contiguous", g, odd_rotations=True)


def append_equals_separate_ops(B, H, cap, pos, n, d, vb, dt, form, g, odd_rotations=False):
    from turboquant_kv import ops
    from turboquant_kv._lib import ops as tops
    Rk, bk, Rv, bv = tables(d, vb)
    nd = torch.float32 if form == "transposed" else dt
    new = lambda *s: torch.randint(0, 256, s, generator=g, device=DEV, dtype=torch.uint8)  # noqa: E731
    kp, vp = new(B, H, cap, d // 2), new(B, H, cap // 64, 8 * vb * d)
    kn, vn = (torch.randn(B, H, cap, generator=g, device=DEV).to(nd) for _ in range(2))
    kv = []
    for _ in range(2):
        x = torch.randn(B, n, H, d, generator=g, device=DEV).to(dt)
        x = x.transpose(1, 2)
        if form == "contiguous":
            x = x.contiguous()
        elif form == "odd":
            buf = torch.empty(x.numel() + 1, dtype=dt, device=DEV)[1:].view(B, H, n, d)
            x = buf.copy_(x)
        kv.append(x)
    want = [t.clone() for t in (kp, kn, vp, vn)]
    for x, R, b, c, nm, bits, val in ((kv[0], Rk, bk, want[0], want[1], 4, False),
                                      (kv[1], Rv, bv, want[2], want[3], vb, True)):
        p, norms = tops().quantize_mse_packed(x.reshape(-1, d), R, b, bits)
        ops.pack_decode_layout(p.view(B * H, n, -1), c.view(B * H, c.shape[2], -1), d, bits, val, pos)
        nm[:, :, pos:pos + n] = norms.view(B, H, n).to(nd)
    if odd_rotations:
        Rk, Rv = (torch.empty(R.numel() + 1, device=DEV)[1:].view(d, d).copy_(R) for R in (Rk, Rv))
    tops().cache_append_dl(kv[0], kv[1], kp, kn, vp, vn, pos, Rk, bk, Rv, bv, 4, vb)
    for got, w, name in zip((kp, kn, vp, vn), want, ("keys", "key norms", "values", "value norms")):
        assert torch.equal(got, w), (name, pos, n, form)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("block,vb", [(16, 2), (16, 3), (16, 4), (32, 2), (64, 2), (64, 3), (64, 4), (128, 3)])
def test_paged_write(block, vb, dt):
    """Slots of prompts (runs from any offset, several sequences in a batch), of decode tokens
    (scattered), padding and out-of-pool slots; pools keep their other tokens."""
    H, nb = 3, 40
    Rk, bk, Rv, bv = tables(64, vb)
    g = torch.Generator(device=DEV).manual_seed(block + vb)
    total = nb * block
    perm = torch.randperm(total, generator=g, device=DEV)
    run = lambda a, n: torch.arange(a, a + n, device=DEV)  # noqa: E731
    pad = torch.tensor([-1, total, total + 5, -7], device=DEV)
    cases = [perm[:1], perm[:48], run(0, 16), run(0, 37), run(7, 100), run(16, 15), run(33, 16),
             torch.cat([run(5, 50), run(320, 40), perm[(perm > 400)][:9]]), torch.cat([run(16, 33), pad]),
             torch.cat([pad, run(48, 64)]), run(0, 32).flip(0),
             torch.cat([run(0, 8), run(24, 24)]), torch.cat([run(3, 13), pad[:1], run(64, 64)])]
    for i, slots in enumerate(cases):
        paged_write_equals_separate_ops(slots, block, vb, dt, H, nb, (Rk, bk, Rv, bv), g, i)


@pytest.mark.parametrize("block,vb", [(16, 3), (32, 4), (64, 2), (64, 3), (64, 4), (128, 3)])
def test_paged_write_large_batches(block, vb):
    """Hundreds of prompts of ragged lengths, more windows of 16 tokens than the launch has waves:
    whole sub-blocks beside single tokens that share their value words, in every half."""
    H, nb, dt = 8, 16384 // block, torch.bfloat16
    g = torch.Generator(device=DEV).manual_seed(block + vb)
    lens = torch.randint(17, 63, (256,), generator=g, device=DEV).tolist()
    starts = torch.randint(0, 40, (256,), generator=g, device=DEV).tolist()
    # 64 slots a sequence, its new tokens from any offset; every fourth one starts anew
    slots = torch.cat([torch.arange(n, device=DEV) + 64 * i + min(a if i % 4 else 0, 64 - n)
                       for i, (n, a) in enumerate(zip(lens, starts))])
    assert slots.numel() // 16 * H > 4096 and slots.unique().numel() == slots.numel()
    paged_write_equals_separate_ops(slots, block, vb, dt, H, nb, tables(64, vb), g, "ragged")
    paged_write_equals_separate_ops(torch.arange(16384, device=DEV), block, vb, dt, H, nb, tables(64, vb), g, "whole")


def paged_write_equals_separate_ops(slots, block, vb, dt, H, nb, tab, g, name):
    from turboquant_kv import ops
    from turboquant_kv._lib import ops as tops
    Rk, bk, Rv, bv = tab
    n = slots.numel()
    k, v = (torch.randn(n, H, 64, generator=g, device=DEV).to(dt) for _ in range(2))
    kp = torch.randint(0, 256, (nb, H, block, 32), generator=g, device=DEV, dtype=torch.uint8)
    shape = (nb, H, block // 64, 512 * vb) if block >= 64 else (nb, H, block // 16, 128 * vb)
    vt = torch.randint(0, 256, shape, generator=g, device=DEV, dtype=torch.uint8)
    kn, vn = (torch.randn(nb, H, block, generator=g, device=DEV) for _ in range(2))
    want = [t.clone() for t in (kp, kn, vt, vn)]
    kq, knew = tops().quantize_mse_packed(k.reshape(-1, 64), Rk, bk, 4)
    vq, vnew = tops().quantize_mse_packed(v.reshape(-1, 64), Rv, bv, vb)
    pairs = torch.empty(n * H, 1, 32, dtype=torch.uint8, device=DEV)
    ops.pack_decode_layout(kq.view(n * H, 1, -1), pairs, 64, 4, False, 0)
    ops.paged_store(pairs.view(n, H, -1), knew.float().view(n, H), slots, want[0], want[1])
    ops.paged_store_value_tiles(vq.view(n, H, -1), vnew.float().view(n, H), slots, want[2], want[3])
    tops().paged_write_dl(k, v, slots, kp, kn, vt, vn, Rk, bk, Rv, bv)
    for got, w, what in zip((kp, kn, vt, vn), want, ("keys", "key norms", "values", "value norms")):
        assert torch.equal(got, w), (what, name)


def test_cache_append_tracked_and_empty():
    """Keys or values with a gradient mark the cache and what is computed from it (a backward says
    that there is none); an append of no tokens is refused in every layout."""
    from turboquant_kv import QuantizedKVCache, TurboQuantConfig
    g = torch.Generator(device=DEV).manual_seed(5)
    k, v = (torch.randn(1, 2, 40, 64, generator=g, device=DEV).bfloat16() for _ in range(2))
    q = torch.randn(1, 4, 64, generator=g, device=DEV).bfloat16()
    make = lambda kb=4: QuantizedKVCache(TurboQuantConfig(key_bits=kb, value_bits=3), 1, 128, 2, 64)  # noqa: E731
    plain, tracked = make(), make()
    plain.append(0, k, v)
    tracked.append(0, k.clone().requires_grad_(), v)
    for a, b in zip((plain._kstore, plain._vstore, plain._key_norms, plain._val_norms),
                    (tracked._kstore, tracked._vstore, tracked._key_norms, tracked._val_norms)):
        assert torch.equal(a[0], b[0])
    assert not plain.decode_attention(0, q).requires_grad
    assert tracked.decode_attention(0, q).requires_grad
    for kb in (4, 3):
        with pytest.raises(RuntimeError):
            make(kb).append(0, k[:, :, :0], v[:, :, :0])
