"""The matrix-core quantizer of bf16 / fp16 rows (csrc/tq_q16.h) against the general kernels (a
wave per row up to 16,384 rows, tiled above), which rows at an odd 2-byte offset take: codes and norms bit for bit, since the
coordinates whose code its sums leave open are summed again in the general kernel's order.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


def rows(n, d, kind, dt, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(n, d, generator=g, device=DEV)
    if kind == "tiny":  # norms below the kernel's regular range, subnormal elements
        x = x * (1e-12 if dt == torch.bfloat16 else 1e-6)
    elif kind == "large":  # some norms overflow the type
        x = x * (1e37 if dt == torch.bfloat16 else 1e4)
    elif kind == "special":
        x[::5] = 0.0
        x[1, 0], x[2, 1], x[3, d - 1] = float("inf"), float("nan"), -float("inf")
        x[4], x[6] = 1e-40, 3e-8
        x[7] = 0.0
        x[7, 3] = -1.0
    return x.to(dt)


def unaligned(x):
    buf = torch.empty(x.numel() + 1, dtype=x.dtype, device=DEV)
    y = buf[1:].view(x.shape)
    y.copy_(x)
    return y


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 128])
def test_rows_equal_general_kernel(d, dt):
    """n around the 16-row tiles, the workgroups and the grid, 1-4 bits; norms that overflow,
    vanish or are NaN; codebooks and rotations of other scales, with equal or unsorted
    boundaries (for which every code is summed in order)."""
    from turboquant_kv._lib import ops
    from turboquant_kv.codebook import lloyd_max_codebook, make_rotation_matrix

    R = make_rotation_matrix(d, 42).to(DEV)
    for bits in (1, 2, 3, 4):
        bnd = lloyd_max_codebook(bits, d)[0].to(DEV)
        cases = [(n, "normal", bnd, R) for n in (1, 15, 16, 17, 127, 129, 70_001)]
        cases += [(515, k, bnd, R) for k in ("tiny", "large", "special")]
        cases += [(515, "normal", b, r) for b, r in
                  ((bnd * 1e-4, R), (bnd[:1].expand_as(bnd).contiguous(), R), (bnd.flip(0).contiguous(), R),
                   (bnd, R * 37.5), (bnd, R * 1e-3))]
        for i, (n, kind, b, r) in enumerate(cases):
            x = rows(n, d, kind, dt, 100 * bits + i)
            p0, n0 = ops().quantize_mse_packed(unaligned(x), r, b, bits)
            p1, n1 = ops().quantize_mse_packed(x, r, b, bits)
            assert torch.equal(p0, p1), (bits, n, kind, i)
            assert n1.dtype == dt and torch.equal(n0.view(torch.int16), n1.view(torch.int16)), (bits, n, kind, i)


@pytest.mark.parametrize("d", [64, 128])
def test_packed_rows_at_any_address(d):
    """Outputs that are not aligned to a plane are stored byte by byte (C ABI)."""
    import numpy as np

    import capi
    from turboquant_kv.codebook import lloyd_max_codebook, make_rotation_matrix

    R = make_rotation_matrix(d, 42).to(DEV)
    x = rows(333, d, "normal", torch.bfloat16, 5)
    for bits in (1, 2, 3, 4):
        bnd = lloyd_max_codebook(bits, d)[0].to(DEV)
        got = []
        for off in (0, 3):
            buf = torch.zeros(333 * bits * d // 8 + 16, dtype=torch.uint8, device=DEV)
            nm = torch.empty(333, device=DEV)
            capi.check(capi.lib().tq_quantize_mse_rows(
                capi.p(x), capi.TQ_BF16, capi.i64(333), capi.i32(d), capi.p(R), capi.p(bnd), capi.i32(bits),
                capi.p(buf[off:]), capi.p(nm), capi.TQ_F32, capi.stream()))
            torch.cuda.synchronize()
            got.append(buf[off: off + 333 * bits * d // 8].cpu().numpy())
            assert not buf[off + 333 * bits * d // 8:].any()
        assert np.array_equal(got[0], got[1]), bits


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 128])
def test_rotation_at_any_address(d, dt):
    """A rotation that is not 16-byte aligned goes to the general kernels, few rows and many."""
    from turboquant_kv._lib import ops
    from turboquant_kv.codebook import lloyd_max_codebook, make_rotation_matrix

    R = make_rotation_matrix(d, 42).to(DEV)
    bnd = lloyd_max_codebook(4, d)[0].to(DEV)
    for n in (1, 300, 16_385):
        x = rows(n, d, "normal", dt, n)
        p0, n0 = ops().quantize_mse_packed(x, R, bnd, 4)
        p1, n1 = ops().quantize_mse_packed(x, unaligned(R), bnd, 4)
        assert torch.equal(p0, p1) and torch.equal(n0.view(torch.int16), n1.view(torch.int16)), n
