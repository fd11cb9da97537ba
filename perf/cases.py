"""The work this package is timed on: index search, quantizing, and attention over packed
KV caches, through the package's public classes.

A case is a dict of plain values; `kind` names the path:

  search    TurboQuantIndex.search over an index built with add()
  quantize  TurboQuantMSE / TurboQuantProd .quantize
  cache     QuantizedKVCache: one decode step (append one token per sequence, attend)
  layer     TurboQuantLayer (the HuggingFace cache's layer): one decode step, either fused
            (attend over the packed history) or not (update returns the dequantized
            history and the new token, for the model's own attention)
  paged     PagedKVPools.forward, the vLLM backend's step: a prefill chunk of `new` tokens
            per sequence, or one decode token per sequence (`new` = 0) with ragged lengths
"""

import math
import os
import random
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "turboquant-kv_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from turboquant_kv import (QuantizedKVCache, TurboQuantConfig, TurboQuantIndex,  # noqa: E402
                           TurboQuantMSE, TurboQuantProd)
from turboquant_kv.hf_integration import TurboQuantLayer, turboquant_attention  # noqa: E402
from turboquant_kv.vllm_plugin import PagedKVPools, TurboQuantAttentionMetadata  # noqa: E402

DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
SIZES = {"float32": 4, "float16": 2, "bfloat16": 2}
CHUNK = 1 << 20  # database rows made at a time
DEV = "cuda"


def _search(name, n, dim, bits, mode, nq, k):
    return dict(name=name, kind="search", n=n, dim=dim, bits=bits, mode=mode, nq=nq, k=k)


def _attn(name, kind, **kw):
    c = dict(name=name, kind=kind, hq=32, hkv=8, dim=64, vbits=2, dtype="bfloat16")
    c.update(kw)
    return c


def listed():
    return [
        # one query over a small collection: a request's latency
        _search("search_65k_q1", 65_536, 128, 4, "mse", 1, 10),
        # one query over a large collection: the benchmark's headline
        _search("search_10m_q1", 10_000_000, 128, 4, "mse", 1, 10),
        # a batch of queries at the default bit width, recall@100 evaluation
        _search("search_1m_q64_b3", 1_000_000, 128, 3, "mse", 64, 100),
        # 200-dim word vectors in the unbiased (QJL) mode, a ragged row count
        _search("search_prod_390k_d200", 390_001, 200, 4, "prod", 16, 10),
        # building an index over a million 128-dim descriptors, QJL mode
        dict(name="quantize_prod_1m", kind="quantize", n=1_000_000, dim=128, bits=4, mode="prod",
             dtype="float32"),
        # a prompt's keys entering a cache: 16-bit rows of 128-dim heads
        dict(name="quantize_bf16_kv", kind="quantize", n=262_147, dim=128, bits=4, mode="mse",
             dtype="bfloat16"),
        # one sequence, a short context: the latency of a decode step's layer
        _attn("cache_b1_1k", "cache", batch=1, context=1000),
        # a batch at long context, 128-dim heads
        _attn("cache_b32_16k_d128", "cache", batch=32, context=16_384, dim=128, vbits=3),
        # the end-to-end decode benchmark's layer: batch 64 after a 4096-token prompt
        _attn("layer_b64_4k", "layer", batch=64, context=4351, vbits=3, fused=True),
        # the HuggingFace cache as a drop-in: the whole history comes back dequantized
        _attn("layer_b8_4k_plain", "layer", batch=8, context=4095, dim=128, vbits=4, fused=False),
        # a 4096-token prompt through the paged backend
        _attn("paged_prefill_4k", "paged", batch=1, context=4096, new=4096, block=16),
        # a serving batch's decode step: ragged contexts in blocks of 16
        _attn("paged_decode_b48", "paged", batch=48, context=8192, new=0, block=16),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["search", "search", "quantize", "cache", "layer", "paged", "paged"])
    if kind == "search":
        dim = rng.choice([64, 128, 128, 200, 100])
        mode = rng.choice(["mse", "mse", "prod"])
        bits = rng.choice([2, 3, 4, 4]) if mode == "mse" else rng.choice([3, 4])
        n = _log(rng, 10_000, 10_000_000 if dim in (64, 128) else 2_000_000)
        # batches of queries: up to the work of 64 queries over a million rows, and of 16
        # over 400k where every query's row scores are summed exactly (prod, other dims)
        pairs = 64e6 if dim in (64, 128) and mode == "mse" else 6e6
        nq = 1 if rng.random() < 0.4 else max(1, _log(rng, 1, max(1.0, min(256.0, pairs / n))))
        return dict(kind=kind, n=n, dim=dim, bits=bits, mode=mode, nq=nq,
                    k=rng.choice([1, 10, 10, 32, 100]))
    if kind == "quantize":
        dim = rng.choice([64, 128, 128, 200])
        mode = rng.choice(["mse", "mse", "prod"])
        dtype = rng.choice(["float32", "bfloat16", "float16"])
        most = 1_000_000 if dtype == "float32" and dim <= 128 else 200_000
        if mode == "prod" and dtype != "float32":
            most = 50_000
        return dict(kind=kind, n=_log(rng, 500, most), dim=dim,
                    bits=rng.choice([2, 3, 4]) if mode == "prod" else rng.choice([1, 2, 3, 4]),
                    mode=mode, dtype=dtype)
    hq, hkv = rng.choice([(32, 8), (32, 8), (8, 8), (28, 4), (16, 2)])
    vbits = rng.choice([2, 3, 4])
    c = dict(kind=kind, hq=hq, hkv=hkv, dim=64, vbits=vbits,
             dtype=rng.choice(["bfloat16", "bfloat16", "float16", "float32"]))
    if kind == "paged":
        c["block"] = rng.choice([16, 16, 32, 64])
        if rng.random() < 0.5:  # a prefill chunk, with or without a history before it
            c["batch"] = rng.choice([1, 1, 2, 4])
            c["new"] = _log(rng, 16, 4096 // c["batch"])
            c["context"] = c["new"] + (0 if rng.random() < 0.5 else
                                       rng.randrange(1, max(2, 4097 - c["new"])))
        else:
            c["batch"], c["new"] = _log(rng, 1, 64), 0
            c["context"] = _log(rng, 100, 8192)
        return c
    c["dim"] = rng.choice([64, 128])
    c["batch"] = _log(rng, 1, 64)
    rows = 1 << 22 if kind == "cache" else 1 << 19  # (sequence, head, token) rows of a layer
    if kind == "layer":
        c["fused"] = rng.random() < 0.5
        rows = 1 << 21 if c["fused"] else 1 << 18
    c["context"] = max(65, min(_log(rng, 100, 32_768), rows // (c["batch"] * hkv)))
    return c


# ------------------------------------------------------------------------------- inputs

def _gen(seed, salt):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 1000 + salt)


def _vectors(case, seed):
    """The database / input rows, CHUNK at a time: unit embeddings, or (prod) non-negative
    heavy-tailed descriptors at 128 dims and log-normally scaled dims elsewhere."""
    g, d = _gen(seed, 1), case["dim"]
    scale = torch.exp(torch.randn(d, generator=g, device=DEV))
    for at in range(0, case["n"], CHUNK):
        x = torch.randn(min(CHUNK, case["n"] - at), d, generator=g, device=DEV)
        if case["mode"] == "mse":
            x = x / x.norm(dim=1, keepdim=True)
        elif d == 128:
            x = x.mul_(40).abs_().floor_().clamp_(0, 255)
        else:
            x = x.mul_(scale)
        yield x


def _rows(case, seed):
    """16-bit rows stand for a cache's keys: a few channels larger than the others."""
    x = torch.cat(list(_vectors(case, seed)))
    if case["dtype"] != "float32":
        x = torch.randn(x.shape, generator=_gen(seed, 2), device=DEV)
        x[:, :: 17] *= 4.0
    return x.to(DTYPES[case["dtype"]])


def _queries(case, seed):
    q = torch.randn(case["nq"], case["dim"], generator=_gen(seed, 3), device=DEV)
    return (q / q.norm(dim=1, keepdim=True)).half()


def _kv(case, seed, salt, *shape):
    """Keys (a few outlier channels) and values of the given leading shape."""
    g, dt, d = _gen(seed, salt), DTYPES[case["dtype"]], case["dim"]
    k = torch.randn(*shape, d, generator=g, device=DEV)
    k[..., :: 17] *= 3.0
    v = torch.randn(*shape, d, generator=g, device=DEV)
    return k.to(dt), v.to(dt)


def _history(case, seed):
    """(first token, keys, values) of a cache's prompt, a few thousand tokens at a time."""
    B, H, T = case["batch"], case["hkv"], case["context"]
    step = max(64, (1 << 27) // (B * H * case["dim"]) // 64 * 64)
    for at in range(0, T, step):
        k, v = _kv(case, seed, 100 + at, B, H, min(step, T - at))
        yield at, k, v


def _step(case, seed):
    """The decode step's query [B, Hq, d] and its token's key and value [B, Hkv, d]."""
    g = _gen(seed, 4)
    q = 1.5 * torch.randn(case["batch"], case["hq"], case["dim"], generator=g, device=DEV)
    k, v = _kv(case, seed, 5, case["batch"], case["hkv"])
    return q.to(DTYPES[case["dtype"]]), k, v


def _lens(case):
    """Context lengths of a paged batch, the new tokens included: ragged for decode."""
    B, T = case["batch"], case["context"]
    if case["new"]:
        return [T] * B
    r = random.Random(B * 100_003 + T)
    return [T] + [r.randint(max(1, T // 8), T) for _ in range(B - 1)]


def _paged(case, seed):
    """Per sequence: keys and values of its whole context [T, Hkv, d]; and the queries of
    the new tokens [tokens, Hq, d]."""
    seqs = [_kv(case, seed, 100 + b, T, case["hkv"]) for b, T in enumerate(_lens(case))]
    n = case["batch"] * max(1, case["new"])
    q = 1.5 * torch.randn(n, case["hq"], case["dim"], generator=_gen(seed, 4), device=DEV)
    return seqs, q.to(DTYPES[case["dtype"]])


def prepare(case, seed):
    kind = case["kind"]
    if kind == "search":
        ix = TurboQuantIndex(case["dim"], case["bits"], mode=case["mode"], device=DEV)
        for x in _vectors(case, seed):
            ix.add(x)
        return dict(case=case, ix=ix, q=_queries(case, seed))
    if kind == "quantize":
        cls = TurboQuantMSE if case["mode"] == "mse" else TurboQuantProd
        return dict(case=case, tq=cls(case["dim"], case["bits"], device=DEV), x=_rows(case, seed))
    cfg = TurboQuantConfig(key_bits=4, value_bits=case["vbits"])
    B, H, T, d = case["batch"], case["hkv"], case["context"], case["dim"]
    if kind == "paged":
        return _prepare_paged(case, seed, cfg)
    q, k, v = _step(case, seed)
    if kind == "cache":
        store = QuantizedKVCache(cfg, 1, T + 1, H, d, device=DEV, batch_size=B)
        for _, hk, hv in _history(case, seed):
            store.append(0, hk, hv)
    else:
        store = TurboQuantLayer(cfg, fused_attention=case["fused"])
        with torch.no_grad():
            hist = list(_history(case, seed))
            hk, hv = torch.cat([h[1] for h in hist], 2), torch.cat([h[2] for h in hist], 2)
            del hist
            store.update(hk, hv)
            store.update(hk[:, :, :1], hv[:, :, :1])  # room for the step's token
    return dict(case=case, store=store, q=q, k=k.unsqueeze(2), v=v.unsqueeze(2))


def _prepare_paged(case, seed, cfg):
    H, bs, B = case["hkv"], case["block"], case["batch"]
    lens, new = _lens(case), max(1, case["new"])
    (seqs, q), nblk = _paged(case, seed), [-(-t // bs) for t in _lens(case)]
    pools = PagedKVPools(cfg, 1, sum(nblk) + 7, bs, H, case["dim"], device=DEV, layout="decode")
    order = torch.randperm(sum(nblk) + 7, generator=_gen(seed, 6), device=DEV)
    tables = torch.zeros(B, max(nblk), dtype=torch.int32, device=DEV)
    slots, keys, vals, used = [], [], [], 0
    for b, (k, v) in enumerate(seqs):
        blocks = order[used: used + nblk[b]]
        used += nblk[b]
        tables[b, : nblk[b]] = blocks.to(torch.int32)
        t = torch.arange(lens[b], device=DEV)
        slot = blocks[t // bs] * bs + t % bs
        old = lens[b] - new
        if old:
            pools.write(0, k[:old], v[:old], slot[:old])
        slots.append(slot[old:]), keys.append(k[old:]), vals.append(v[old:])
    starts = [b * new for b in range(B + 1)]
    md = TurboQuantAttentionMetadata(
        slot_mapping=torch.cat(slots), seq_lens=torch.tensor(lens, dtype=torch.int32, device=DEV),
        block_tables=tables, query_start_loc=torch.tensor(starts, dtype=torch.int32, device=DEV),
        num_prefills=B if case["new"] else 0, query_start_loc_cpu=starts, seq_lens_cpu=lens)
    return dict(case=case, pools=pools, md=md, q=q, k=torch.cat(keys), v=torch.cat(vals))


# ---------------------------------------------------------------------------------- run

def run(state):
    case, kind = state["case"], state["case"]["kind"]
    scale = 1.0 / math.sqrt(case["dim"])
    if kind == "search":
        return list(state["ix"].search(state["q"], k=case["k"]))
    if kind == "quantize":
        return list(state["tq"].quantize(state["x"]))
    with torch.no_grad():
        if kind == "paged":
            pools = state["pools"]
            out = pools.forward(state["q"], state["k"], state["v"], state["md"], scale)
            return dict(out=out, **pools.layers[0])
        store = state["store"]
        if kind == "cache":
            store.seq_lens[0] = case["context"]  # the step's token is written anew
            store.append(0, state["k"], state["v"])
            return [store.decode_attention(0, state["q"], scale)]
        store.seq_len = case["context"]
        k, v = store.update(state["k"], state["v"])
        if not case["fused"]:
            return [k, v]
        out, _ = turboquant_attention(None, state["q"].unsqueeze(2), k, v, None, scale)
        return dict(out=out, kp=store.kp, kn=store.kn, vp=store.vp, vn=store.vn)


# --------------------------------------------------------------------------------- work

def work(case):
    d, kind = case["dim"], case["kind"]
    bpp = (d + 7) // 8
    if kind == "search":
        row = case["bits"] * bpp + (8 if case["mode"] == "prod" else 4)
        terms = 4 if case["mode"] == "prod" else 2  # codes, and signs
        return {"bytes": case["n"] * row + case["nq"] * (2 * d + 12 * case["k"]),
                "flops": terms * case["n"] * case["nq"] * d}
    if kind == "quantize":
        sz, prod = SIZES[case["dtype"]], case["mode"] == "prod"
        return {"bytes": case["n"] * (sz * d + case["bits"] * bpp + sz * (2 if prod else 1)),
                "flops": case["n"] * 2 * d * d * (3 if prod else 1)}
    sz, hq, hkv = SIZES[case["dtype"]], case["hq"], case["hkv"]
    row = (4 + case["vbits"]) * bpp  # a token's codes of one head
    if kind == "paged":
        lens, new = _lens(case), max(1, case["new"])
        io = case["batch"] * new * (2 * hq + 2 * hkv) * d * sz
        seen = sum(sum(range(t - new + 1, t + 1)) for t in lens)
        return {"bytes": sum(lens) * hkv * (row + 8) + io,
                "flops": 4 * d * hq * seen + 4 * d * d * case["batch"] * new * hkv}
    rows = case["batch"] * hkv * (case["context"] + 1)
    norm = 4 if kind == "cache" else sz
    if kind == "layer" and not case["fused"]:  # history in, history and new token out
        return {"bytes": rows * (row + 2 * norm + 2 * d * sz), "flops": 4 * d * d * rows}
    io = case["batch"] * (2 * hq + 2 * hkv) * d * sz
    return {"bytes": rows * (row + 2 * norm) + io,
            "flops": 4 * d * (hq // hkv) * rows + 4 * d * d * case["batch"] * (hq + hkv)}


def tolerance(case):
    kind = case["kind"]
    if kind == "search":
        # fp32 scores; ids differ where two scores are within a rounding of each other
        return {"rel": 2e-6, "differ": 2e-3}
    if kind == "quantize":
        # codes at a decision boundary depend on the order of the rotation's sums: a few in
        # a million in fp32, and one in thousands where 16-bit outputs are rounded first
        if case["dtype"] == "float32":
            return {"rel": 1e-6, "max": 1e-4, "differ": 2e-4}
        return {"rel": 1e-3, "max": 0.02, "differ": 5e-3}
    # attention and dequantized rows: the output type's rounding (seen: 2e-3 in bfloat16,
    # 3e-4 in float16), in fp32 the odd code at a boundary (up to 5e-5 of an attention
    # output, 3e-4 of the rows themselves); the caches' own bytes differ as quantize's do
    plain = kind == "layer" and not case["fused"]
    rel = {"float32": 2e-3 if plain else 5e-4, "float16": 3e-3, "bfloat16": 1e-2}[case["dtype"]]
    return {"rel": rel, "max": 0.9 if plain else 40 * rel, "differ": 2e-3}


# -------------------------------------------------------------------------------- exact

def _rotation(d, seed):
    """QR of a Gaussian matrix, signs fixed: the float32 matrix itself is the input."""
    q, r = np.linalg.qr(np.random.RandomState(seed).randn(d, d).astype(np.float32))
    s = np.sign(np.diag(r))
    s[s == 0] = 1.0
    return torch.from_numpy(np.ascontiguousarray(q * s[None, :])).to(DEV)


def _codebook(bits, d):
    """Lloyd-Max centroids and midpoints of N(0, 1/d): at most 200 steps from 2^bits evenly
    spaced points on [-3, 3]."""
    c = list(np.linspace(-3.0, 3.0, 1 << bits))
    cdf = lambda t: 0.5 * math.erfc(-t / math.sqrt(2.0))  # noqa: E731
    pdf = lambda t: math.exp(-0.5 * t * t) / math.sqrt(2.0 * math.pi)  # noqa: E731
    for _ in range(200):
        b = [-math.inf] + [0.5 * (p + q) for p, q in zip(c, c[1:])] + [math.inf]
        new = [(pdf(lo) - pdf(hi)) / (cdf(hi) - cdf(lo)) for lo, hi in zip(b, b[1:])]
        if max(abs(p - q) for p, q in zip(c, new)) < 1e-12:
            break
        c = new
    c = np.array(c)
    b = 0.5 * (c[:-1] + c[1:])
    f32 = lambda a: torch.tensor(a / math.sqrt(d), dtype=torch.float32, device=DEV)  # noqa: E731
    return f32(b), f32(c)


def _quantize64(x, R, bits):
    """(codes, norms, unit rows) of x [n, d] in 64 bits; 16-bit inputs round the norm, the
    unit rows, the operands and the rotated rows to their type, as the method defines."""
    dt = x.dtype
    rd = (lambda t: t) if dt == torch.float32 else (lambda t: t.to(dt).double())
    bnd, _ = _codebook(bits, x.shape[1])
    x = x.double()
    n = rd(x.square().sum(1).sqrt())
    u = rd(x / n.clamp(min=1e-10)[:, None])
    y = rd(u @ rd(R.double()).t())
    return torch.bucketize(y, rd(bnd.double())), n, u


def _dequantized(x, bits, seed, dtype=torch.float32, lead=None):
    """x [.., d] quantized and reconstructed in 64 bits (operands rounded to dtype)."""
    shape, d = x.shape, x.shape[-1]
    R, c = _rotation(d, seed), _codebook(bits, d)[1]
    out = torch.empty(x.numel() // d, d, dtype=torch.float64, device=DEV)
    flat = x.reshape(-1, d)
    for at in range(0, flat.shape[0], CHUNK):
        codes, n, _ = _quantize64(flat[at: at + CHUNK], R, bits)
        out[at: at + CHUNK] = (c.to(dtype).double()[codes] @ R.to(dtype).double()) * n[:, None]
    return out.view(shape)


def _attend(q, k, v, visible=None):
    """softmax(q k^T / sqrt(d)) v for q [Hq, n, d] over k, v [Hkv, T, d], in 64 bits."""
    G = q.shape[0] // k.shape[0]
    out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
    for h in range(q.shape[0]):
        s = (q[h].double() @ k[h // G].t().contiguous()) / math.sqrt(q.shape[-1])
        if visible is not None:
            s = s.masked_fill(~visible, float("-inf"))
        out[h] = torch.softmax(s, -1) @ v[h // G]
    return out


def _exact_search(case, seed):
    d, prod, q = case["dim"], case["mode"] == "prod", _queries(case, seed).double()
    bits = case["bits"] - prod
    R, c = _rotation(d, 42), _codebook(bits, d)[1].double()
    if prod:
        S = torch.randn(d, d, generator=torch.Generator().manual_seed(42 + 12345)).to(DEV).double()
    best = torch.empty(case["nq"], 0, dtype=torch.float64, device=DEV)
    for x in _vectors(case, seed):
        parts = []
        for rows in x.split(CHUNK // 4):
            codes, n, u = _quantize64(rows, R, bits)
            rec = c[codes] @ R.double()
            if prod:
                r = u - rec
                sign = torch.where(r @ S.t() >= 0, 1.0, -1.0).double()
                rec = rec + math.sqrt(math.pi / 2) / d * r.norm(dim=1, keepdim=True) * (sign @ S)
            parts.append((q @ rec.t().contiguous()) * n[None])
        s = torch.cat([best] + parts, 1)
        best = torch.topk(s, min(case["k"], s.shape[1]), dim=1).values
    return [best, None]


def exact(case, seed):
    kind = case["kind"]
    if kind == "search":
        return _exact_search(case, seed)
    d = case["dim"]
    if kind == "quantize":
        x = _rows(case, seed)
        n = torch.cat([r.double().square().sum(1).sqrt() for r in x.split(CHUNK // 4)])
        if case["mode"] == "mse":
            return [None, n]
        if case["dtype"] != "float32":
            return [None, None, None, n]
        R, c = _rotation(d, 42), _codebook(case["bits"] - 1, d)[1].double()
        res = []
        for r in x.split(CHUNK // 4):
            codes, _, u = _quantize64(r, R, case["bits"] - 1)
            res.append((u - c[codes] @ R.double()).norm(dim=1))
        return [None, None, torch.cat(res), n]
    if kind == "paged":
        seqs, q = _paged(case, seed)
        new, out = max(1, case["new"]), torch.empty(q.shape, dtype=torch.float64, device=DEV)
        for b, (k, v) in enumerate(seqs):
            T = k.shape[0]
            k = _dequantized(k.transpose(0, 1).contiguous(), 4, 42)
            v = _dequantized(v.transpose(0, 1).contiguous(), case["vbits"], 43)
            vis = torch.arange(T, device=DEV)[None] <= torch.arange(T - new, T, device=DEV)[:, None]
            out[b * new: (b + 1) * new] = _attend(q[b * new: (b + 1) * new].transpose(0, 1), k, v,
                                                  vis).transpose(0, 1)
        return dict(out=out, kn=None, kp=None, vn=None, vt=None)
    q, nk, nv = _step(case, seed)
    ks, vs = [], []
    plain = kind == "layer" and not case["fused"]
    dt = DTYPES[case["dtype"]] if plain else torch.float32
    for _, k, v in _history(case, seed):
        ks.append(_dequantized(k, 4, 42, dt))
        vs.append(_dequantized(v, case["vbits"], 43, dt))
    nk, nv = nk.unsqueeze(2), nv.unsqueeze(2)
    if kind == "cache":  # the step's own token is read back from the cache
        ks.append(_dequantized(nk, 4, 42))
        vs.append(_dequantized(nv, case["vbits"], 43))
    else:
        ks.append(nk.double())
        vs.append(nv.double())
    k, v = torch.cat(ks, 2), torch.cat(vs, 2)
    del ks, vs
    if plain:
        return [k, v]
    out = torch.stack([_attend(q[b].unsqueeze(1), k[b], v[b])[:, 0] for b in range(case["batch"])])
    if kind == "cache":
        return [out]
    return dict(out=out.unsqueeze(1), kp=None, kn=None, vp=None, vn=None)
