"""PagedKVPools.forward's prefill rows: written by the kernel in the result's type, equal to
the fp32 result converted once, also where the result is a given tensor, an unaligned one or
the queries' own memory."""
import pytest
import torch

from turboquant_kv.config import TurboQuantConfig

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32, torch.float64])
@pytest.mark.parametrize("how", ["none", "given", "unaligned", "alias"])
def test_forward_prefill_rows(dtype, how):
    from turboquant_kv.vllm_plugin import PagedKVPools, TurboQuantAttentionMetadata
    hkv, hq, d, bs, lens = 2, 6, 64, 16, [97, 33]
    pools = PagedKVPools(TurboQuantConfig(), 1, 16, bs, hkv, d, DEV, layout="decode")
    g = torch.Generator(device=DEV).manual_seed(3)
    n = sum(lens)
    tables = torch.randperm(16, generator=g, device=DEV).to(torch.int32).view(2, 8)
    slots = torch.cat([tables[i].long()[torch.arange(t, device=DEV) // bs] * bs + torch.arange(t, device=DEV) % bs
                       for i, t in enumerate(lens)])
    q, k, v = (torch.randn(n, h, d, generator=g, device=DEV).to(dtype) for h in (hq, hkv, hkv))
    md = TurboQuantAttentionMetadata(
        num_prefills=2, slot_mapping=slots, block_tables=tables,
        seq_lens=torch.tensor(lens, dtype=torch.int32, device=DEV),
        query_start_loc=torch.tensor([0, lens[0], n], dtype=torch.int32, device=DEV))
    out = None
    if how == "given":
        out = torch.empty_like(q)
    elif how == "unaligned":
        out = torch.empty(q.numel() + 1, dtype=dtype, device=DEV)[1:].view_as(q)
    pools.write(0, k, v, slots)
    want = torch.cat([pools.prefill(0, q[a:b], tables[i], b - a, 0.125).to(dtype)
                      for i, (a, b) in enumerate([(0, lens[0]), (lens[0], n)])])
    if how == "alias":
        out = q
    got = pools.forward(q, k, v, md, 0.125, output=out)
    if out is not None:
        assert got.data_ptr() == out.data_ptr()
    assert got.dtype == dtype and torch.equal(got, want)  # the same sums, converted once


def test_forward_keeps_graph_and_strides():
    """Through queries with a gradient a prefill's result is a node of the graph (whose backward says
    that there is none); a decode step's result has the strides of dense queries in another order."""
    from turboquant_kv.vllm_plugin import PagedKVPools, TurboQuantAttentionMetadata
    pools = PagedKVPools(TurboQuantConfig(), 1, 4, 16, 2, 64, DEV, layout="decode")
    g = torch.Generator(device=DEV).manual_seed(3)
    q, k, v = (torch.randn(20, h, 64, generator=g, device=DEV).bfloat16() for h in (4, 2, 2))
    table = torch.arange(4, device=DEV, dtype=torch.int32).view(1, 4)

    def step(query, n, t, npf):
        md = TurboQuantAttentionMetadata(
            num_prefills=npf, slot_mapping=torch.arange(t - n, t, device=DEV), block_tables=table,
            seq_lens=torch.tensor([t], dtype=torch.int32, device=DEV),
            query_start_loc=torch.tensor([0, n], dtype=torch.int32, device=DEV))
        return pools.forward(query, k[:n], v[:n], md, 0.125)

    plain = step(q, 20, 20, 1)
    tracked = step(q.clone().requires_grad_(), 20, 20, 1)
    assert tracked.requires_grad and not plain.requires_grad and torch.equal(plain, tracked.detach())
    one = q[:1]
    other = one.transpose(1, 2).contiguous().transpose(1, 2)
    a, b = step(one, 1, 21, 0), step(other, 1, 21, 0)
    assert torch.equal(a, b) and b.stride() == other.stride() != a.stride()


def test_forward_under_vmap():
    """A prefill and a decode step mapped over batches of queries."""
    from turboquant_kv.vllm_plugin import PagedKVPools, TurboQuantAttentionMetadata
    pools = PagedKVPools(TurboQuantConfig(), 1, 4, 16, 2, 64, DEV, layout="decode")
    g = torch.Generator(device=DEV).manual_seed(3)
    q, k, v = (torch.randn(2, 20, h, 64, generator=g, device=DEV).bfloat16() for h in (4, 2, 2))
    for n, t, npf in ((20, 20, 1), (1, 21, 0)):
        md = TurboQuantAttentionMetadata(
            num_prefills=npf, slot_mapping=torch.arange(t - n, t, device=DEV),
            block_tables=torch.arange(4, device=DEV, dtype=torch.int32).view(1, 4),
            seq_lens=torch.tensor([t], dtype=torch.int32, device=DEV),
            query_start_loc=torch.tensor([0, n], dtype=torch.int32, device=DEV),
            query_start_loc_cpu=[0, n], seq_lens_cpu=[t])
        step = lambda x: pools.forward(x, k[0, :n], v[0, :n], md, 0.125)  # noqa: E731
        want = torch.stack([step(q[0, :n]), step(q[1, :n])])
        assert torch.equal(torch.vmap(step)(q[:, :n]), want)
