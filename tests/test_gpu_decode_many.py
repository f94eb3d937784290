"""Paged decode of more sequences than a wavefront has lanes: token chunks sized from the actual lengths, four sequences a lane."""
from __future__ import annotations

import random

import pytest
import torch

from flashquant_amd import kernels as K, load_native
from oracle import tq_oracle as O
from tests.gpu_util import book

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _lens(n, ctx, kind):
    r = random.Random(n)
    if kind == "alike":
        return [ctx] * n
    if kind == "ragged":
        return [ctx] + [r.randint(1, ctx) for _ in range(n - 1)]
    return [0 if s % 5 == 3 else r.choice((1, 64, ctx - 1, ctx, ctx)) for s in range(n)]      # some without a key


def _worst_row(got, want):
    """The worst row's relative error (2-norms over the last dimension)."""
    got, want = got.double().flatten(0, -2), want.double().flatten(0, -2)
    return ((got - want).norm(dim=1) / want.norm(dim=1)).max().item()


# A row against the oracle's, or against the same row in other chunks: the merged row and the one rotated back are rounded to the
# query type, 2^-8 (bf16) or 2^-11 of a value at most on either side, weights, keys and values in fp16 add 2^-11 each.
LIMIT = {torch.bfloat16: 4 * 2 ** -8, torch.float16: 8 * 2 ** -11}


def _inputs(n, hq, hkv, d, bs, ctx, dtype, row_bytes, norm_at):
    """Random packed bytes with norms around sqrt(d), pages in random order, queries; all on the GPU."""
    g = torch.Generator(device=DEV).manual_seed(n + ctx)
    pages = (ctx + bs - 1) // bs
    cache = torch.randint(0, 256, (n * pages, bs, row_bytes), dtype=torch.uint8, generator=g, device=DEV)
    rows = cache.view(-1, row_bytes)
    for at, size in norm_at:
        rows[:, at:at + 4 * hkv] = (size * d ** 0.5 * (0.5 + torch.rand(rows.shape[0], hkv, generator=g, device=DEV))).view(torch.uint8)
    table = torch.randperm(n * pages, generator=g, device=DEV).view(n, pages).int()
    return g, cache, table, torch.randn(n, hq, d, generator=g, device=DEV).to(dtype)


def _tq4_inputs(n, hq, hkv, d, bs, ctx, dtype):
    half = hkv * d // 2
    return _inputs(n, hq, hkv, d, bs, ctx, dtype, hkv * (d + 8), ((half, 1.0), (2 * half + 4 * hkv, 1.0)))


# sequences around a wavefront's worth and around whole groups of four of them, chunks of at least 384 rows (of one token, of 2,
# 4 and 8), the split counts that leave more than a round of workgroups; the last three keep the fixed chunks
@pytest.mark.parametrize("kind", ["alike", "ragged", "sparse"])
@pytest.mark.parametrize("n,hq,hkv,d,splits,ctx", [(65, 8, 8, 128, 5, 1700), (130, 32, 8, 128, 2, 700), (201, 8, 8, 128, 3, 1000), (256, 8, 8, 128, 2, 700),
                                                   (90, 8, 4, 128, 4, 2700), (131, 8, 2, 128, 2, 2600), (129, 8, 1, 128, 2, 5200), (70, 4, 4, 256, 4, 1400),
                                                   (140, 32, 16, 64, 2, 700), (67, 8, 1, 256, 4, 3300), (257, 8, 8, 128, 2, 700), (97, 8, 1, 128, 3, 300)])
def test_decode_of_many_sequences(n, hq, hkv, d, splits, ctx, kind):
    """Against the same sequences sixty at a time (the path that the other tests hold against the oracle).  Either rounds the
    merged row and the rotated one to bf16 (half of 2^-7 of a value at most, each), after weights in fp16 (2^-11): one part in fifty
    of a value, or of 1 where that is larger."""
    lens, bs = _lens(n, ctx, kind), 16
    c, _, r = book(d)
    g = torch.Generator(device=DEV).manual_seed(n)
    pages = (ctx + bs - 1) // bs
    cache = torch.randint(0, 256, (n * pages, bs, hkv * (d + 8)), dtype=torch.uint8, generator=g, device=DEV)
    rows, half = cache.view(-1, hkv * (d + 8)), hkv * d // 2
    for at in (half, 2 * half + 4 * hkv):                                # the norms of the keys, of the values
        norms = d ** 0.5 * (0.5 + torch.rand(rows.shape[0], hkv, generator=g, device=DEV))
        rows[:, at:at + 4 * hkv] = norms.view(torch.uint8)
    table = torch.randperm(n * pages, generator=g, device=DEV).view(n, pages).int()
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    q = torch.randn(n, hq, d, generator=g, device=DEV).to(torch.bfloat16)
    rest = (c.to(DEV), c.to(DEV), r.to(DEV), hkv, d, bs)
    got = K.split_k_paged_decode(q, cache, table, sl, *rest, num_splits=splits, out=torch.full_like(q, 7.0)).float()
    want = torch.cat([K.split_k_paged_decode(q[s:s + 60], cache, table[s:s + 60], sl[s:s + 60], *rest, num_splits=splits).float()
                      for s in range(0, n, 60)])
    assert ((got - want).abs() <= 2e-2 * want.abs().clamp(min=1.0)).all()
    assert _worst_row(got[sl > 0], want[sl > 0]) <= LIMIT[torch.bfloat16]
    assert (got[sl == 0] == 0).all()


# one group of 8 KV heads and two, rows of 8, 4 and 2 tokens, 64 coordinates; chunks of 384 to 1024 rows; more live pairs than CUs
# ("alike"), or fewer
STEPS = [(70, 8, 8, 128, 16, torch.bfloat16, 4, 1700), (130, 16, 16, 128, 8, torch.float16, 2, 900), (65, 8, 8, 128, 32, torch.float16, 4, 4000),
         (96, 8, 1, 128, 16, torch.bfloat16, 3, 9300), (129, 4, 2, 128, 32, torch.float16, 3, 4100), (131, 16, 4, 128, 16, torch.bfloat16, 2, 1700),
         (201, 32, 8, 64, 16, torch.float16, 2, 1700), (256, 8, 8, 128, 16, torch.bfloat16, 2, 700)]


@pytest.mark.parametrize("kind", ["alike", "ragged", "sparse"])
@pytest.mark.parametrize("n,hq,hkv,d,bs,dtype,splits,ctx", STEPS)
def test_serving_step_of_many_sequences(n, hq, hkv, d, bs, dtype, splits, ctx, kind):
    """The new token is stored by whichever workgroup the sized chunks give the end of its sequence: every stored row is the
    oracle's (an index may be its neighbour where the coordinate lies on the boundary in float32), no other byte changes, and
    the output is the oracle's over the cache that the step left."""
    lens = _lens(n, ctx, kind)
    c, b, r = (t.to(DEV) for t in book(d))
    g, cache, table, q = _tq4_inputs(n, hq, hkv, d, bs, ctx, dtype)
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    key, value = (torch.randn(n, hkv, d, generator=g, device=DEV).to(dtype) for _ in range(2))
    last = (sl.long() - 1).clamp(min=0)
    slots = table.long()[torch.arange(n, device=DEV), last // bs] * bs + last % bs
    stored = (sl > 0) & (torch.arange(n, device=DEV) % 7 != 3)              # some sequences store nothing
    slots = torch.where(stored, slots, -1)
    got_cache = cache.clone()
    got = K.tq4_store_and_decode(key, value, slots, q, got_cache, table, sl, c, c, r, b, hkv, d, bs, num_splits=splits,
                                 out=torch.full_like(q, 7.0))
    rows, before = got_cache.view(-1, hkv * (d + 8)), cache.view(-1, hkv * (d + 8))
    keep = torch.ones(rows.shape[0], dtype=torch.bool, device=DEV)
    keep[slots[stored]] = False
    assert torch.equal(rows[keep], before[keep])
    side = hkv * (d // 2 + 4)
    for at, x in ((0, key), (side, value)):
        x = x[stored].double()
        norm = x.norm(dim=-1)
        y = (x / (norm[..., None] + 1e-10)) @ r.double().T
        packed = rows[slots[stored], at:at + hkv * d // 2]
        index = torch.stack((packed >> 4, packed & 15), dim=-1).view(-1, hkv, d).long()
        want_index = torch.bucketize(y, b.double())
        off = (index - want_index).abs()
        gap = (y[..., None] - b.double()).abs().amin(dim=-1)
        assert off.max() <= 1 and (gap[off > 0] <= 1e-6).all()
        got_norm = rows[slots[stored], at + hkv * d // 2:at + side].contiguous().view(torch.float32)
        assert ((got_norm.double() - norm) / norm).abs().max() <= 2e-6
    with torch.device(DEV):
        want = O.split_k_paged_decode(q, got_cache, table, sl, c, c, r, hkv, d, bs)
    assert _worst_row(got[sl > 0], want[sl > 0]) <= LIMIT[dtype]
    assert (got[sl == 0] == 0).all()


@pytest.mark.parametrize("kind", ["alike", "ragged", "sparse"])
@pytest.mark.parametrize("n,hq,hkv,bs,dtype,splits,ctx", [(66, 32, 8, 16, torch.bfloat16, 5, 2500), (130, 16, 16, 8, torch.float16, 2, 900),
                                                          (256, 8, 8, 32, torch.bfloat16, 2, 1100)])
def test_prod_decode_of_many_sequences(n, hq, hkv, bs, dtype, splits, ctx, kind):
    """3-bit + sign keys, against the oracle.  The sketched query in fp16 beside the rotated one: one part in 2^11 more."""
    d, native = 128, load_native()
    kn, kg, _, vn, row_bytes = K.prod_page_layout(hkv, d)
    c3, c4, r = book(d, 3)[0].to(DEV), book(d)[0].to(DEV), book(d)[2].to(DEV)
    sketch = native.qjl_matrix(d, 42).to(DEV)
    g, cache, table, q = _inputs(n, hq, hkv, d, bs, ctx, dtype, row_bytes, ((kn, 1.0), (kg, 0.185), (vn, 1.0)))
    sl = torch.tensor(_lens(n, ctx, kind), dtype=torch.int32, device=DEV)
    got = K.prod_paged_decode(q, cache, table, sl, c3, c4, r, sketch, hkv, d, bs, num_splits=splits, out=torch.full_like(q, 7.0))
    with torch.device(DEV):
        want = O.prod_paged_decode(q, cache, table, sl, c3, c4, r, sketch, hkv, d, bs)
    assert _worst_row(got[sl > 0], want[sl > 0]) <= LIMIT[dtype] + 2 ** -11
    assert (got[sl == 0] == 0).all()


@pytest.mark.parametrize("hq,hkv,splits,ctx", [(8, 8, 4, 1700), (8, 1, 3, 9300)])
def test_captured_step_of_many_sequences_over_other_lengths(hq, hkv, splits, ctx):
    """The chunks follow from the lengths at the replay, not at the capture: every replay is the eager step, bit for bit."""
    C = load_native()
    n, d, bs, dtype = 96, 128, 16, torch.bfloat16
    c, b, r = (t.to(DEV) for t in book(d))
    ev, od = (t.to(DEV).contiguous() for t in O.split_rotation(r.cpu()))
    g, cache, table, q = _tq4_inputs(n, hq, hkv, d, bs, ctx, dtype)
    key, value = (torch.randn(n, hkv, d, generator=g, device=DEV).to(dtype) for _ in range(2))
    sl = torch.tensor(_lens(n, ctx, "sparse"), dtype=torch.int32, device=DEV)
    slots = torch.full((n,), -1, dtype=torch.int64, device=DEV)
    ws = torch.empty(C.paged_decode_workspace_bytes(n, hq, hkv, d, bs, table.shape[1], splits), dtype=torch.uint8, device=DEV)
    cache_g, out_g = cache.clone(), torch.empty_like(q)

    def step(cache_t, out_t):
        C.tq4_store_and_decode(key, value, slots, ev, od, b, q, cache_t, table, sl, c, c, r, hkv, d, bs, None, out_t, splits, ws)

    step(cache_g, out_g)                                   # first call outside the capture (runtime set-up)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step(cache_g, out_g)
    for kind in ("alike", "ragged", "sparse", "alike"):
        sl.copy_(torch.tensor(_lens(n, ctx, kind), dtype=torch.int32))
        last = (sl.long() - 1).clamp(min=0)
        slots.copy_(torch.where(sl > 0, table.long()[torch.arange(n, device=DEV), last // bs] * bs + last % bs, -1))
        q.copy_(torch.randn(q.shape, generator=g, device=DEV))
        cache_e, out_e = cache_g.clone(), torch.empty_like(q)
        graph.replay()
        torch.cuda.synchronize()
        step(cache_e, out_e)
        torch.cuda.synchronize()
        assert torch.equal(out_g, out_e) and torch.equal(cache_g, cache_e), kind


@pytest.mark.parametrize("kind", ["alike", "ragged", "sparse"])
def test_ring_kernel_with_many_sequences(kind):
    """The ring kernel takes its chunks from the same search as the staged one."""
    C, (n, hq, hkv, d, bs, splits, ctx) = load_native(), (130, 32, 8, 128, 16, 3, 2500)
    c, _, r = (t.to(DEV) for t in book(d))
    _, cache, table, q = _tq4_inputs(n, hq, hkv, d, bs, ctx, torch.bfloat16)
    sl = torch.tensor(_lens(n, ctx, kind), dtype=torch.int32, device=DEV)
    old = C.set_option("decode_ring", 1)
    try:
        got = K.split_k_paged_decode(q, cache, table, sl, c, c, r, hkv, d, bs, num_splits=splits, out=torch.full_like(q, 7.0))
    finally:
        C.set_option("decode_ring", old)
    with torch.device(DEV):
        want = O.split_k_paged_decode(q, cache, table, sl, c, c, r, hkv, d, bs)
    assert _worst_row(got[sl > 0], want[sl > 0]) <= LIMIT[torch.bfloat16]
    assert (got[sl == 0] == 0).all()


# rows (sequences x query heads) on both sides of where 4, 2 and 1 workgroups (16, 8 and 4 at 256 coordinates) share the columns of
# a group of rows, the last group not full; one split, one chunk of splits and several
@pytest.mark.parametrize("splits", [2, 9, 21])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d,hq,hkv,n", [(128, 8, 8, 1), (128, 7, 1, 3), (128, 32, 8, 8), (128, 24, 8, 11), (128, 8, 2, 64), (128, 24, 8, 22),
                                        (256, 8, 8, 1), (256, 7, 1, 9), (256, 16, 4, 4), (256, 6, 2, 11), (256, 8, 1, 16), (256, 12, 4, 11),
                                        (256, 16, 4, 16), (256, 16, 4, 17)])
def test_workgroups_that_share_the_columns_of_a_row(d, hq, hkv, n, dtype, splits):
    """Against the same merged rows rotated by other groupings of rows, columns and contraction: the rows are exact operands and
    the matrix keeps 22 bits, so the float32 sums differ by their order alone, 2^-20 of the row's norm, and what is stored by one
    rounding to the query type more."""
    ctx, bs = 900, 16
    c, _, r = (t.to(DEV) for t in book(d))
    _, cache, table, q = _tq4_inputs(n, hq, hkv, d, bs, ctx, dtype)
    sl = torch.tensor([0 if s == 5 else ctx - 37 * s % 800 for s in range(n)], dtype=torch.int32, device=DEV)
    for rot in (r.contiguous(), r.t().contiguous().t()):                    # row-major and column-major
        rest = (cache, table, sl, c, c, rot, hkv, d, bs)
        got = K.split_k_paged_decode(q, *rest, num_splits=splits, out=torch.full_like(q, 7.0)).double()
        for rows in ((16,) if d == 128 else (4, 8)):
            C = load_native()
            old = C.set_option("reduce_rows", rows)
            try:
                want = K.split_k_paged_decode(q, *rest, num_splits=splits).double()
            finally:
                C.set_option("reduce_rows", old)
            near = 2.0 ** (-7 if dtype == torch.bfloat16 else -10) * want.abs() + 2.0 ** -20 * want.norm(dim=-1, keepdim=True)
            assert ((got - want).abs() <= near).all(), rows
        assert (got[sl == 0] == 0).all() and got[sl > 0].norm(dim=-1).min() > 0
