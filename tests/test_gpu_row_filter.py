"""The filtered row scan (csrc/tq_row_filter.h) against the exact scan: with the workspace of
tq_scan_workspace_bytes the same entry points score every row exactly, with that of
tq_scan_rows_workspace_bytes they filter.  Ids and scores agree bit for bit."""

import ctypes

import pytest
import torch

import capi

pytestmark = pytest.mark.gpu

DEV = "cuda"


def database(N, d, bits, prod, pairs, seed):
    from turboquant_kv._lib import ops
    from turboquant_kv.codebook import lloyd_max_codebook, make_qjl_matrix, make_rotation_matrix
    cb = bits - prod
    R, S = make_rotation_matrix(d, 42).to(DEV), make_qjl_matrix(d, d, 42).to(DEV)
    bnd, cen = (t.to(DEV) for t in lloyd_max_codebook(cb, d))
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(N, d, generator=g, device=DEV) * torch.exp(torch.randn(N, 1, generator=g, device=DEV) * 0.3)
    x[100:140] = x[7]  # exact ties
    x[5] = 0.0
    if prod:
        p, sg, rn, nm = ops().quantize_prod_packed(x, R, bnd, cen, S, bits)
    else:
        (p, nm), sg, rn = ops().quantize_mse_packed(x, R, bnd, bits), None, None
    if pairs:
        p = ops().pack_pair_rows(p, cb, d)
    return dict(p=p, sg=sg, rn=rn, nm=nm, cen=cen, R=R, S=S, bits=bits, prod=prod, pairs=pairs, d=d, N=N)


def random_rows(N, d, bits, prod, seed):
    """A database of random codes: any bytes are rows."""
    from turboquant_kv.codebook import lloyd_max_codebook, make_qjl_matrix, make_rotation_matrix
    g = torch.Generator(device=DEV).manual_seed(seed)
    byte = lambda w: torch.randint(0, 256, (N, w), generator=g, device=DEV, dtype=torch.uint8)  # noqa: E731
    nm = torch.exp(torch.randn(N, generator=g, device=DEV) * 0.3)
    bpp = (d + 7) // 8
    return dict(p=byte((bits - prod) * bpp), sg=byte(bpp) if prod else None, rn=nm * 0.3 if prod else None, nm=nm,
                cen=lloyd_max_codebook(bits - prod, d)[1].to(DEV), R=make_rotation_matrix(d, 42).to(DEV),
                S=make_qjl_matrix(d, d, 42).to(DEV), bits=bits, prod=prod, pairs=0, d=d, N=N)


def scan(db, q, k, filtered):
    Q, N, d, bits = q.shape[0], db["N"], db["d"], db["bits"]
    L, c = capi.lib(), capi
    L.tq_scan_rows_workspace_bytes.restype = ctypes.c_size_t
    small = L.tq_scan_workspace_bytes(c.i64(Q), c.i32(d), c.i32(bits), c.i64(N), c.i32(k))
    big = L.tq_scan_rows_workspace_bytes(c.i64(Q), c.i32(d), c.i32(bits), c.i64(N), c.i32(k),
                                         c.i32(db["prod"]), c.i32(db["pairs"]))
    ws = torch.full((big if filtered else small,), 0xab, dtype=torch.uint8, device=DEV)
    s = torch.empty(Q, k, device=DEV)
    i = torch.empty(Q, k, dtype=torch.long, device=DEV)
    dt = {torch.float32: c.TQ_F32, torch.float16: c.TQ_F16, torch.bfloat16: c.TQ_BF16}[q.dtype]
    tail = (c.i32(bits), c.i32(k), c.p(s), c.p(i), c.p(ws), ctypes.c_size_t(ws.numel()), c.stream())
    head = (c.p(q), dt, c.i64(Q), c.i32(d), c.p(db["p"]))
    if db["prod"]:
        f = L.tq_ip_scan_topk_prod_pair_rows if db["pairs"] else L.tq_ip_scan_topk_prod
        c.check(f(*head, c.p(db["sg"]), c.p(db["rn"]), c.p(db["nm"]), c.i64(N), c.p(db["cen"]), c.p(db["R"]),
                  c.p(db["S"]), *tail))
    else:
        c.check(L.tq_ip_scan_topk(*head, c.p(db["nm"]), c.i64(N), c.p(db["cen"]), c.p(db["R"]), *tail))
    # the exact scan writes its lists, at byte 256 of the workspace, for the queries it answers
    return s, i, big > small, filtered and not bool((ws[256:small] != 0xab).any())


def same(db, q, k, unflagged=False):
    s0, i0, _, _ = scan(db, q, k, False)
    s1, i1, filters, alone = scan(db, q, k, True)
    assert torch.equal(s0.view(torch.int32), s1.view(torch.int32)) and torch.equal(i0, i1), (db["N"], q.shape, k)
    assert alone or not unflagged, (db["N"], q.shape, k)
    return filters


@pytest.mark.parametrize("d", [16, 20, 37, 64, 100, 128, 200, 225, 256])
def test_equals_exact_scan(d):
    """Dims around the 32-dim steps and byte counts, 2-4 bits, with and without signs, row counts
    around the 64-row groups and the table's end, 1 to 33 queries, k from 1 to 128, ties."""
    hit = 0
    for n, (bits, prod) in enumerate(((2, 0), (3, 0), (4, 0), (3, 1), (4, 1))):
        for N in (8192, 8193 + 62 * (n % 2), 20_011):
            db = database(N, d, bits, prod, 0, 10 * d + n)
            g = torch.Generator(device=DEV).manual_seed(d + n)
            for Q, k, dt in ((1, 10, torch.float16), (5, 1, torch.float32), (17, 128, torch.bfloat16),
                             (33, 32, torch.float16)):
                hit += same(db, torch.randn(Q, d, generator=g, device=DEV).to(dt), k)
    assert hit >= 40


@pytest.mark.parametrize("d,bits,prod,N", [(200, 4, 1, 300_007), (100, 3, 0, 300_007), (128, 4, 0, 300_007),
                                           (16, 2, 0, 1_100_003), (37, 3, 1, 1_100_003), (64, 4, 1, 1_100_003)])
def test_several_groups_per_wave(d, bits, prod, N):
    """Row counts at which a wave takes one group after another, its next rows on their way, and
    the sample is spread over the table (its stride above 1; two groups a bucket above 1,048,576)."""
    db = random_rows(N, d, bits, prod, d)
    db["p"][5000:5040] = db["p"][7].clone()  # ties
    db["nm"][5000:5040] = db["nm"][7].clone()
    g = torch.Generator(device=DEV).manual_seed(d)
    for Q, k in ((17, 10), (5, 100)):
        assert same(db, torch.randn(Q, d, generator=g, device=DEV).half(), k, unflagged=True)


def test_rounds_of_queries():
    """More queries than one round of lists holds."""
    db = database(9000, 100, 3, 0, 0, 1)
    q = torch.randn(600, 100, generator=torch.Generator(device=DEV).manual_seed(2), device=DEV)
    assert same(db, q, 10)


@pytest.mark.parametrize("d,bits", [(64, 3), (64, 4), (128, 3), (128, 4)])
def test_prod_pair_rows(d, bits):
    """Prod rows whose codes are pair rows, from where they are filtered."""
    for N in (120_000, 200_033):
        db = database(N, d, bits, 1, 1, d + bits)
        g = torch.Generator(device=DEV).manual_seed(bits)
        for Q, k in ((64, 10), (40, 100), (130, 33)):
            assert same(db, torch.randn(Q, d, generator=g, device=DEV).half(), k)


@pytest.mark.parametrize("N,k", [(28_000_001, 100), (80_000_001, 32)])
def test_lists_hold_large_tables(N, k):
    """The listed rows fit the merge however many rows there are: no query goes on to the exact scan."""
    db = random_rows(N, 16, 2, 0, k)
    assert same(db, torch.randn(3, 16, generator=torch.Generator(device=DEV).manual_seed(k), device=DEV), k, True)


@pytest.mark.parametrize("d", [64, 100, 128])
def test_as_many_results_as_groups(d):
    """128 results from 128 64-row groups, the least rows that are filtered, and one row more."""
    for N in (8192, 8193):
        for bits, prod in ((2, 0), (4, 0), (3, 1)):
            q = torch.randn(16, d, generator=torch.Generator(device=DEV).manual_seed(d), device=DEV)
            assert same(database(N, d, bits, prod, 0, d), q, 128, unflagged=True)


@pytest.mark.parametrize("d,bits,N,nq,k", [(128, 4, 1_000_000, 4, 1), (64, 4, 1_000_000, 6, 2), (64, 2, 1_000_000, 4, 1)])
def test_few_results_around_a_million_rows_scan_exactly(d, bits, N, nq, k):
    """Calls that the exact scan answers faster ask for its workspace only."""
    c, L = capi, capi.lib()
    L.tq_scan_rows_workspace_bytes.restype = ctypes.c_size_t
    size = lambda n, q, kk, prod=0, pairs=0: L.tq_scan_rows_workspace_bytes(  # noqa: E731
        c.i64(q), c.i32(d), c.i32(bits), c.i64(n), c.i32(kk), c.i32(prod), c.i32(pairs))
    base = lambda n, q, kk: L.tq_scan_workspace_bytes(q, d, bits, n, kk)  # noqa: E731
    assert size(N, nq, k) == base(N, nq, k)
    assert size(N, nq, 32) > base(N, nq, 32) and size(N // 10, nq, k) > base(N // 10, nq, k)
    for n, kk, on in ((12_000, 1, False), (12_000, 10, False), (12_000, 32, True), (100_000, 1, True)):
        assert (size(n, 700, kk) > base(n, 700, kk)) == on, (n, kk)  # many queries over few rows
    if d == 64 and bits == 4:  # prod pair rows
        assert size(12_000, 700, 10, 1, 1) == base(12_000, 700, 10)
        assert size(10_000_000, 2, 10, 1, 1) == base(10_000_000, 2, 10)
        assert size(10_000_000, 3, 10, 1, 1) == base(10_000_000, 3, 10)
        assert size(10_000_000, 2, 100, 1, 1) > base(10_000_000, 2, 100)


def test_matrices_at_any_address():
    """A rotation and QJL matrix that are not 16-byte aligned."""
    db = database(9000, 100, 4, 1, 0, 5)
    q = torch.randn(5, 100, generator=torch.Generator(device=DEV).manual_seed(6), device=DEV)
    s0, i0, _, _ = scan(db, q, 10, True)
    for key, off in (("R", 1), ("S", 3)):
        m = db[key]
        db[key] = torch.empty(m.numel() + off, device=DEV)[off:].view(m.shape).copy_(m)
    assert same(db, q, 10, unflagged=True)
    s1, i1, _, _ = scan(db, q, 10, True)
    assert torch.equal(s0, s1) and torch.equal(i0, i1)


@pytest.mark.parametrize("prod", [0, 1])
def test_special_values(prod):
    """Zero, infinite and NaN queries, norms and residual norms, and a database of equal rows: the
    queries the filter cannot bound are answered by the exact scan."""
    db = database(9000, 200, 4, prod, 0, 3)
    g = torch.Generator(device=DEV).manual_seed(4)
    q = torch.randn(18, 200, generator=g, device=DEV)
    q[1], q[2] = 0.0, q[2] * 1e-30
    q[3, 5], q[4, 7] = float("inf"), float("nan")
    q[5] *= 1e30
    assert same(db, q, 10)
    db["nm"][::97], db["nm"][50], db["nm"][51] = -1.0, float("inf"), float("nan")
    if prod:
        db["rn"][60], db["rn"][61] = float("inf"), float("nan")
    assert same(db, q, 100)
    for key in ("p", "sg", "rn", "nm"):
        if db[key] is not None:
            db[key][:] = db[key][7].clone()
    assert same(db, q, 10)
