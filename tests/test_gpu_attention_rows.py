"""How the attention kernels rotate, store and split their query rows: edges of the 32-row blocks,
either layout of the rotation matrix, outputs that are not 16-byte aligned."""
from __future__ import annotations

import pytest
import torch

from flashquant_amd import kernels as K
from oracle import tq_oracle as O
from tests.gpu_util import book, build_paged_case

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 128), (8, 2, 64)])
def test_paged_prefill_output_at_any_alignment(hq, hkv, d, dtype):
    """The rows leave in 16-byte stores where the output allows it and in 2-byte stores where it does not: the
    same bits, and nothing written outside the rows."""
    ql, kv, bs = [33, 1, 64, 0, 31], [33, 70, 200, 9, 31], 16
    c, _, r = book(d)
    _, cache, table, sl = build_paged_case(kv, hq, hkv, d=d, bs=bs, seed=5, dtype=dtype)
    q = torch.randn(sum(ql), hq, d, generator=torch.Generator().manual_seed(6)).to(dtype).to(DEV)
    cu = torch.tensor([0] + list(torch.tensor(ql).cumsum(0)), dtype=torch.int32).to(DEV)
    args = (cu, max(ql), cache.to(DEV), table.to(DEV), sl.to(DEV), c.to(DEV), c.to(DEV))
    want = K.paged_tq4_prefill(q, *args, r.to(DEV), hkv, d, bs)
    for shift in (1, 4):
        room = torch.full((q.numel() + 16,), 7.0, dtype=dtype, device=DEV)
        K.paged_tq4_prefill(q, *args, r.to(DEV), hkv, d, bs, out=room[shift:shift + q.numel()].view_as(q))
        torch.cuda.synchronize()
        assert torch.equal(room[shift:shift + q.numel()].view_as(q), want)
        assert (room[:shift] == 7).all() and (room[shift + q.numel():] == 7).all()
    other = K.paged_tq4_prefill(q, *args, r.t().contiguous().to(DEV).t(), hkv, d, bs)      # the matrix in the other layout
    assert torch.equal(other, want)


def _close(got, want, dtype):
    """bf16 rounds to 2^-9 and fp16 to 2^-12 of a value; the rows are rounded at most three times (query, result, output)
    and keys and weights are held in fp16: three roundings' 2-norm, doubled."""
    rel = (got.cpu().double() - want.double()).norm() / want.double().norm()
    limit = 2 * 3 ** 0.5 * (2 ** -9 if dtype == torch.bfloat16 else 2 ** -11)
    assert rel <= limit, f"relative error {rel:.2e}, limit {limit:.2e}"


def _packed(b, h, n, d, seed):
    c, bnd, r = book(d)
    g = torch.Generator().manual_seed(seed)
    out = []
    for _ in range(2):
        p, m = O.compress(torch.randn(b * h * n, 1, d, generator=g), r, bnd)
        out += [p.reshape(b, h, n, d // 2), m.reshape(b, h, n, 1)]
    return out, c, r


# (batch, query heads, KV heads, queries, keys): one query, a few, more than one 32-row block, more than one workgroup of
# queries, more pieces than one chunk of eight, key counts at and around multiples of a tile
SPLIT = [(1, 8, 2, 1, 448, 128), (1, 8, 2, 1, 449, 128), (1, 4, 1, 3, 513, 64), (1, 8, 1, 2, 511, 256),   # the shortest that are split
         (4, 32, 8, 1, 2500, 128), (1, 8, 2, 1, 1024, 128), (1, 8, 8, 1, 6001, 64), (2, 8, 1, 5, 4097, 128), (1, 16, 2, 33, 2111, 64),
         (1, 5, 1, 130, 4160, 128), (1, 8, 1, 17, 1023, 64), (1, 4, 4, 2, 16384, 128)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,hq,hkv,nq,nkv,d", SPLIT)
def test_attention_over_split_contexts(b, hq, hkv, nq, nkv, d, dtype):
    """Few workgroups over long contexts: the keys run in pieces, combined by a second launch."""
    kv, c, r = _packed(b, hkv, nkv, d, 31)
    q = torch.randn(b, hq, nq, d, generator=torch.Generator().manual_seed(32)).to(dtype)
    want = O.fused_tq_attention(q, *kv, c, c, r)
    got = K.fused_tq_attention(q.to(DEV), *[t.to(DEV) for t in kv], c.to(DEV), c.to(DEV), r.to(DEV))
    _close(got, want, dtype)


@pytest.mark.parametrize("d", [64, 128])
def test_attention_over_split_contexts_causal_and_huge_norms(d):
    """Causal rows that see nothing of a piece, and rows whose norms exceed fp16 in one piece only."""
    kv, c, r = _packed(1, 2, 2500, d, 41)
    kv[1][:, :, 2000:2003] *= 1e-3
    kv[3][:, :, 2100] *= 4000.0
    q = torch.randn(1, 8, 2400, d, generator=torch.Generator().manual_seed(42)).to(torch.bfloat16)
    for n in (40, 2400):
        want = O.fused_tq_attention(q[:, :, :n], *kv, c, c, r, is_causal=n > 40)
        got = K.fused_tq_attention(q[:, :, :n].contiguous().to(DEV), *[t.to(DEV) for t in kv], c.to(DEV), c.to(DEV), r.to(DEV), is_causal=n > 40)
        _close(got, want, torch.bfloat16)


# (queries, keys) per sequence: a mixed batch with long single queries, chunks of one and of several workgroups on long
# contexts, idle sequences and sequences without keys, more sequences than a wavefront has lanes
BATCHES = [([1, 1, 40, 300, 0, 1], [3000, 17, 2000, 300, 9, 1500]), ([130, 70], [4000, 2500]), ([1], [4001]), ([64, 0], [64, 0]),
           ([1 + (s % 3) * 20 for s in range(70)], [1 + (s % 3) * 20 + (s % 7) * 90 for s in range(70)]),
           ([1] * 5, [0, 1, 64, 65, 2048])]


@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 128), (16, 2, 64), (5, 1, 128)])
@pytest.mark.parametrize("batch", range(len(BATCHES)))
def test_paged_prefill_order_and_split(batch, hq, hkv, d):
    """Work is handed out longest first and long contexts of few queries in pieces: every row of every sequence is written
    once, whatever the mixture (rows of sequences without keys are zero)."""
    ql, kv = BATCHES[batch]
    bs, dtype = 16, torch.bfloat16
    c, _, r = book(d)
    _, cache, table, sl = build_paged_case(kv, hq, hkv, d=d, bs=bs, seed=51, dtype=dtype)
    q = torch.randn(sum(ql), hq, d, generator=torch.Generator().manual_seed(52)).to(dtype)
    cu = torch.tensor([0] + list(torch.tensor(ql).cumsum(0)), dtype=torch.int32)
    for causal in (True, False):
        want = O.paged_prefill(q, cu, cache, table, sl, c, c, r, hkv, d, bs, causal=causal)
        out = torch.full_like(q, 7.0).to(DEV)
        K.paged_tq4_prefill(q.to(DEV), cu.to(DEV), max(ql), cache.to(DEV), table.to(DEV), sl.to(DEV), c.to(DEV), c.to(DEV),
                            r.to(DEV), hkv, d, bs, causal=causal, out=out)
        _close(out, want, dtype)
        for s, n in enumerate(kv):
            if n == 0:
                assert (out[int(cu[s]):int(cu[s + 1])] == 0).all()


def test_split_attention_under_capture():
    """The split call allocates from the caching allocator and launches twice: replays give the eager result."""
    kv, c, r = _packed(1, 8, 3000, 128, 61)
    dev = [t.to(DEV) for t in kv]
    cd, rd = c.to(DEV), r.to(DEV)
    q = torch.randn(1, 32, 1, 128, generator=torch.Generator().manual_seed(62)).to(torch.bfloat16).to(DEV)
    K.fused_tq_attention(q, *dev, cd, cd, rd)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = K.fused_tq_attention(q, *dev, cd, cd, rd)
    for k in range(4):
        q.copy_(torch.randn(q.shape, generator=torch.Generator().manual_seed(63 + k)).to(q.dtype))
        eager = K.fused_tq_attention(q, *dev, cd, cd, rd)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)


# (batch, query heads, KV heads, queries, keys, causal): one row, the edges of the 32-row blocks and of the 32-key tiles, fewer
# and more rows than a workgroup has, an odd number of heads per KV head, contexts in pieces
WIDE = [(1, 1, 1, 1, 1, False), (1, 4, 1, 31, 31, True), (2, 4, 2, 32, 33, True), (1, 8, 2, 33, 65, False), (1, 3, 1, 97, 97, True),
        (1, 16, 4, 300, 300, True), (2, 8, 1, 1, 3001, False), (1, 8, 2, 5, 1055, False), (1, 4, 2, 130, 2049, False)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,hq,hkv,nq,nkv,causal", WIDE)
def test_head_dim_256_rows(b, hq, hkv, nq, nkv, causal, dtype):
    kv, c, r = _packed(b, hkv, nkv, 256, 71)
    if nkv > 40:                                       # norms beyond fp16's range in some rows of one tile
        kv[1][:, :, 35:38] *= 1e-3
        kv[3][:, :, 36] *= 4000.0
    q = torch.randn(b, hq, nq, 256, generator=torch.Generator().manual_seed(72)).to(dtype)
    want = O.fused_tq_attention(q, *kv, c, c, r, is_causal=causal)
    dev = [t.to(DEV) for t in (q, *kv, c, c, r)]
    room = K.fused_tq_attention(*dev, is_causal=causal)
    _close(room, want, dtype)
    other = K.fused_tq_attention(*dev[:-1], r.t().contiguous().to(DEV).t(), is_causal=causal)      # the matrix in the other layout
    assert torch.equal(other, room)


@pytest.mark.parametrize("hq,hkv", [(8, 2), (5, 1)])
@pytest.mark.parametrize("batch", range(len(BATCHES)))
def test_paged_prefill_order_and_split_head_dim_256(batch, hq, hkv):
    test_paged_prefill_order_and_split(batch, hq, hkv, 256)


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("b,hq,hkv,nq,nkv,causal", [(4, 16, 8, 390, 2111, False), (1, 8, 1, 4201, 4201, True)])
def test_prompts_in_pieces(b, hq, hkv, nq, nkv, causal, d):
    """Enough workgroups of whole prompts in pieces for the combine launch that works like the attention workgroups; the last
    workgroup of a sequence with fewer than eight units, the last unit with fewer than 32 rows."""
    kv, c, r = _packed(b, hkv, nkv, d, 81)
    q = torch.randn(b, hq, nq, d, generator=torch.Generator().manual_seed(82)).to(torch.float16)
    want = O.fused_tq_attention(q, *kv, c, c, r, is_causal=causal)
    got = K.fused_tq_attention(q.to(DEV), *[t.to(DEV) for t in kv], c.to(DEV), c.to(DEV), r.to(DEV), is_causal=causal)
    _close(got, want, torch.float16)


@pytest.mark.parametrize("d", [64, 128, 256])
def test_paged_prompts_in_pieces(d):
    ql, kv, hq, hkv, bs = [390, 7, 260, 300], [2100, 1500, 260, 1031], 16, 8, 16
    c, _, r = book(d)
    _, cache, table, sl = build_paged_case(kv, hq, hkv, d=d, bs=bs, seed=91, dtype=torch.bfloat16)
    q = torch.randn(sum(ql), hq, d, generator=torch.Generator().manual_seed(92)).to(torch.bfloat16)
    cu = torch.tensor([0] + list(torch.tensor(ql).cumsum(0)), dtype=torch.int32)
    want = O.paged_prefill(q, cu, cache, table, sl, c, c, r, hkv, d, bs, causal=True)
    got = K.paged_tq4_prefill(q.to(DEV), cu.to(DEV), max(ql), cache.to(DEV), table.to(DEV), sl.to(DEV), c.to(DEV), c.to(DEV),
                              r.to(DEV), hkv, d, bs)
    _close(got, want, torch.bfloat16)
