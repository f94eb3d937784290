"""How the attention kernels rotate, store and split their query rows: edges of the 32-row blocks,
either layout of the rotation matrix, outputs that are not 16-byte aligned."""
from __future__ import annotations

import pytest
import torch

from flashquant_amd import kernels as K
from oracle import tq_oracle as O
from tests.gpu_util import (attention_in_one_piece, attention_on_packed_rows, attention_workspace_bytes, book, build_paged_case,
                            prefill_in_one_piece, prefill_on_packed_rows)

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
    packed = prefill_on_packed_rows(q, *args[:-1], r.to(DEV), hkv, d, bs)                  # (keys and values not expanded)
    for shift in (1, 4):
        for same in (want, packed):
            room = torch.full((q.numel() + 16,), 7.0, dtype=dtype, device=DEV)
            out = room[shift:shift + q.numel()].view_as(q)
            if same is want:
                K.paged_tq4_prefill(q, *args, r.to(DEV), hkv, d, bs, out=out)
            else:
                prefill_on_packed_rows(q, *args[:-1], r.to(DEV), hkv, d, bs, out=out)
            torch.cuda.synchronize()
            assert torch.equal(out, same)
            assert (room[:shift] == 7).all() and (room[shift + q.numel():] == 7).all()
    other = K.paged_tq4_prefill(q, *args, r.t().contiguous().to(DEV).t(), hkv, d, bs)      # the matrix in the other layout
    assert torch.equal(other, want)


def _close(got, want, dtype):
    """The 2-norm of a rounding's error is below 2^-9 (bf16; 2^-9.4 for values spread evenly over a binade) or 2^-12 (fp16) of
    the values'.  bf16: the rows are rounded at most three times (query, result, output).  fp16: keys and values are too, and
    the weights towards zero (2^-11), (5 + 4)^(1/2) * 2^-12 in all.  Doubled; the worst of thousands of rows: doubled again."""
    got, want = got.cpu().double().flatten(0, -2), want.double().flatten(0, -2)
    limit = 2 * (3 ** 0.5 * 2 ** -9 if dtype == torch.bfloat16 else 3 * 2 ** -12)
    rel = (got - want).norm() / want.norm()
    assert rel <= limit, f"relative error {rel:.2e}, limit {limit:.2e}"
    live = want.norm(dim=1) > 0
    _rows_close(got[live], want[live], 2 * limit)


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
SPLIT = [(1, 8, 2, 1, 449, 128), (1, 4, 1, 3, 705, 64), (1, 8, 1, 2, 449, 256), (1, 8, 1, 2, 511, 256),   # the shortest that are split
         (4, 32, 8, 1, 2500, 128), (1, 8, 2, 1, 1024, 128), (1, 8, 8, 1, 6001, 64), (2, 8, 1, 5, 4097, 128), (1, 16, 2, 33, 2111, 64),
         (1, 5, 1, 130, 4160, 128), (1, 8, 1, 17, 1023, 64), (1, 4, 4, 2, 16384, 128)]
NOT_SPLIT = [(1, 8, 2, 1, 448, 128), (1, 4, 1, 3, 513, 64)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,hq,hkv,nq,nkv,d", SPLIT + NOT_SPLIT)
def test_attention_over_split_contexts(b, hq, hkv, nq, nkv, d, dtype):
    """Few workgroups over long contexts: the keys run in pieces, combined by a second launch."""
    kv, c, r = _packed(b, hkv, nkv, d, 31)
    q = torch.randn(b, hq, nq, d, generator=torch.Generator().manual_seed(32)).to(dtype)
    want = O.fused_tq_attention(q, *kv, c, c, r)
    got = K.fused_tq_attention(q.to(DEV), *[t.to(DEV) for t in kv], c.to(DEV), c.to(DEV), r.to(DEV))
    _close(got, want, dtype)


# query heads that four do not divide, more than one workgroup of 8 units a KV head, a group of rows with one query and with two;
# as many groups as still leave CUs for several workgroups each (b = 1, 2) and more (b = 40)
@pytest.mark.parametrize("d", [128, 256])
@pytest.mark.parametrize("b,hq,hkv,nq", [(1, 1, 1, 1), (2, 6, 2, 2), (1, 5, 1, 1), (2, 7, 1, 2), (1, 9, 1, 1), (1, 12, 1, 2), (2, 16, 1, 1), (1, 18, 2, 2),
                                         (1, 6, 2, 3), (2, 5, 1, 6), (40, 5, 1, 1), (40, 3, 1, 2)])
def test_heads_that_share_a_group_of_combined_rows(b, hq, hkv, nq, d):
    kv, c, r = _packed(b, hkv, 640, d, 33)
    q = torch.randn(b, hq, nq, d, generator=torch.Generator().manual_seed(34)).to(torch.bfloat16)
    want = O.fused_tq_attention(q, *kv, c, c, r)
    dev = [t.to(DEV) for t in (q, *kv, c, c, r)]
    got = K.fused_tq_attention(*dev)
    _close(got, want, torch.bfloat16)
    assert torch.equal(K.fused_tq_attention(*dev[:-1], r.t().contiguous().to(DEV).t()), got)       # the matrix in the other layout


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
        # the prompt of 2400 runs on expanded keys: here in pieces on the packed ones
        _close(attention_on_packed_rows(q[:, :, :n].contiguous().to(DEV), *[t.to(DEV) for t in kv], c.to(DEV), r.to(DEV), is_causal=n > 40), want,
               torch.bfloat16)


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
        packed = prefill_on_packed_rows(q.to(DEV), cu.to(DEV), max(ql), cache.to(DEV), table.to(DEV), sl.to(DEV), c.to(DEV), r.to(DEV), hkv, d,
                                        bs, causal=causal, out=torch.full_like(q, 7.0).to(DEV))
        for got in (out, packed):
            _close(got, want, dtype)
            for s, n in enumerate(kv):
                if n == 0:
                    assert (got[int(cu[s]):int(cu[s + 1])] == 0).all()


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
    _close(attention_on_packed_rows(*dev[:5], *dev[6:], is_causal=causal), want, dtype)


@pytest.mark.parametrize("hq,hkv", [(8, 2), (5, 1)])
@pytest.mark.parametrize("batch", range(len(BATCHES)))
def test_paged_prefill_order_and_split_head_dim_256(batch, hq, hkv):
    test_paged_prefill_order_and_split(batch, hq, hkv, 256)


WHOLE_PROMPTS = [(4, 16, 8, 390, 2111, False), (1, 8, 1, 4201, 4201, True)]


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("b,hq,hkv,nq,nkv,causal", WHOLE_PROMPTS)
def test_prompts_in_pieces(b, hq, hkv, nq, nkv, causal, d):
    """Enough workgroups of whole prompts in pieces for the combine launch that works like the attention workgroups; the last
    workgroup of a sequence with fewer than eight units, the last unit with fewer than 32 rows."""
    kv, c, r = _packed(b, hkv, nkv, d, 81)
    q = torch.randn(b, hq, nq, d, generator=torch.Generator().manual_seed(82)).to(torch.float16)
    want = O.fused_tq_attention(q, *kv, c, c, r, is_causal=causal)
    got = K.fused_tq_attention(q.to(DEV), *[t.to(DEV) for t in kv], c.to(DEV), c.to(DEV), r.to(DEV), is_causal=causal)
    _close(got, want, torch.float16)
    # (with room for its expanded keys the causal prompt takes no part of this kernel)
    _close(attention_on_packed_rows(q.to(DEV), *[t.to(DEV) for t in kv], c.to(DEV), r.to(DEV), is_causal=causal), want, torch.float16)


@pytest.mark.parametrize("d", [64, 128, 256])
def test_paged_prompts_in_pieces(d):
    ql, kv, hq, hkv, bs = [390, 7, 260, 300], [2100, 1500, 260, 1031], 16, 8, 16
    c, _, r = book(d)
    _, cache, table, sl = build_paged_case(kv, hq, hkv, d=d, bs=bs, seed=91, dtype=torch.bfloat16)
    q = torch.randn(sum(ql), hq, d, generator=torch.Generator().manual_seed(92)).to(torch.bfloat16)
    cu = torch.tensor([0] + list(torch.tensor(ql).cumsum(0)), dtype=torch.int32)
    want = O.paged_prefill(q, cu, cache, table, sl, c, c, r, hkv, d, bs, causal=True)
    args = (q.to(DEV), cu.to(DEV), max(ql), cache.to(DEV), table.to(DEV), sl.to(DEV), c.to(DEV))
    got = K.paged_tq4_prefill(*args, c.to(DEV), r.to(DEV), hkv, d, bs)
    _close(got, want, torch.bfloat16)
    _close(prefill_on_packed_rows(*args, r.to(DEV), hkv, d, bs), want, torch.bfloat16)


# (batch, query heads, KV heads, queries, keys): rows for the combine launch by 4 and by 16 rows, and enough workgroups for
# the one that works like the attention's workgroups
IN_PIECES = [(1, 8, 2, 2, 2111), (1, 8, 2, 40, 2111), (4, 16, 8, 390, 2111)]
# what is wrong with the inputs, and whether every row of the first KV head shows it
POISON = {"query nan": False, "query inf": False, "key norm nan": True, "key norm inf": True, "all key norms nan": True,
          "far key norm nan": True, "value norm nan": True, "value norm inf": True}


def _poison(kind, kn, vn, row):
    """NaN and infinities in the norms (tokens, any shape behind: views of the first KV head) or in the query row."""
    nan, inf = float("nan"), float("inf")
    if kind == "query nan":
        row[5] = nan
    elif kind == "query inf":
        row[5] = inf
    elif kind == "key norm nan":
        kn[1500] = nan
    elif kind == "key norm inf":
        kn[700] = inf
    elif kind == "all key norms nan":
        kn[:] = nan
    elif kind == "far key norm nan":            # in a piece whose weights are nothing beside the others'
        kn[:] *= 40
        kn[0:250] *= 1e-6
        kn[3] = nan
    elif kind == "value norm nan":
        vn[10] = nan
    elif kind == "value norm inf":
        vn[2000] = inf


def _check_poisoned(got, one_piece, clean, everywhere, row, heads):
    """`got` has no number where the run in one piece has none; rows of other KV heads (and other rows than the poisoned
    query) are the clean ones.  (rows of `heads`, D) tensors."""
    got, one_piece, clean = (t.float() for t in (got, one_piece, clean))
    assert torch.equal(got.isfinite(), one_piece.isfinite())
    bad = ~got.isfinite()
    if everywhere:
        assert bad[:heads].all()
    else:
        assert bad[0, row].all()
        bad = bad.clone()
        bad[0, row] = False
        assert not bad.any()
        ok = got.isfinite()
        assert torch.equal(got[ok], clean[ok])
    assert torch.equal(got[heads:], clean[heads:])


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("kind", list(POISON))
@pytest.mark.parametrize("b,hq,hkv,nq,nkv", IN_PIECES)
def test_nan_and_inf_stay_visible_in_pieces(b, hq, hkv, nq, nkv, kind, d):
    """A row whose scores, weights or values are no numbers is no number either, in pieces as in one."""
    assert attention_workspace_bytes(b, nq, nkv, hq, hkv, d) > 0
    kv, c, r = _packed(b, hkv, nkv, d, 95)
    q = torch.randn(b, hq, nq, d, generator=torch.Generator().manual_seed(96)).to(torch.bfloat16).to(DEV)
    kv, c, r = [t.to(DEV) for t in kv], c.to(DEV), r.to(DEV)
    clean = K.fused_tq_attention(q, *kv, c, c, r)
    _poison(kind, kv[1][0, 0], kv[3][0, 0], q[0, 0, 1])
    got = K.fused_tq_attention(q, *kv, c, c, r)
    want = attention_in_one_piece(q, *kv, c, r)
    if "far" in kind:
        clean[0, :hq // hkv] = got[0, :hq // hkv]
    _check_poisoned(*(t.flatten(0, 1) for t in (got, want, clean)), POISON[kind], 1, hq // hkv)


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("kind", list(POISON))
@pytest.mark.parametrize("ql,kv,hq,hkv", [([2, 1], [2111, 1800], 8, 2), ([390, 260, 300, 350], [2111, 2100, 2048, 2050], 16, 8)])
def test_nan_and_inf_stay_visible_in_pieces_paged(ql, kv, hq, hkv, kind, d):
    bs = 16
    assert attention_workspace_bytes(len(ql), max(ql), max(kv), hq, hkv, d) > 0
    c, _, r = book(d)
    _, cache, table, sl = build_paged_case(kv, hq, hkv, d=d, bs=bs, seed=97, dtype=torch.bfloat16)
    q = torch.randn(sum(ql), hq, d, generator=torch.Generator().manual_seed(98)).to(torch.bfloat16).to(DEV)
    cu = torch.tensor([0] + list(torch.tensor(ql).cumsum(0)), dtype=torch.int32).to(DEV)
    cache, table, sl, c, r = (t.to(DEV) for t in (cache, table, sl, c, r))
    args = (cu, max(ql), cache, table, sl, c)
    def prefill():                                                  # as the operator runs it, and in pieces on the packed rows
        return (K.paged_tq4_prefill(q, *args, c, r, hkv, d, bs, causal=False), prefill_on_packed_rows(q, *args, r, hkv, d, bs, causal=False))

    cleans = prefill()
    pos = torch.arange(kv[0])
    slots = table[0].long().cpu()[pos // bs] * bs + pos % bs
    norms = cache.view(-1, hkv * (d + 8)).view(torch.float32)
    kn, vn = norms[slots, hkv * d // 8], norms[slots, hkv * (d + 4) // 4]
    _poison(kind, kn, vn, q[1, 0])
    norms[slots, hkv * d // 8], norms[slots, hkv * (d + 4) // 4] = kn, vn
    want = prefill_in_one_piece(q, *args, r, hkv, d, bs, causal=False)
    first = lambda t: t[:ql[0]].transpose(0, 1)                     # noqa: E731  (heads, rows of the first sequence, D)
    for got, clean in zip(prefill(), cleans):
        if "far" in kind:
            clean[:ql[0], :hq // hkv] = got[:ql[0], :hq // hkv]
        _check_poisoned(first(got), first(want), first(clean), POISON[kind], 1, hq // hkv)
        assert torch.equal(got[ql[0]:], clean[ql[0]:])


@pytest.mark.parametrize("d", [64, 128, 256])
def test_nan_stays_where_it_is_seen_in_causal_prompts(d):
    """Rows in front of a NaN key see nothing of it, the others are no numbers: in pieces as in one."""
    n, key = 4201, 2500
    assert attention_workspace_bytes(1, n, n, 8, 1, d, prompts=True) > 0
    kv, c, r = _packed(1, 1, n, d, 99)
    kv[1][..., key, :] = float("nan")
    q = torch.randn(1, 8, n, d, generator=torch.Generator().manual_seed(100)).to(torch.bfloat16).to(DEV)
    kv, c, r = [t.to(DEV) for t in kv], c.to(DEV), r.to(DEV)
    for got in (K.fused_tq_attention(q, *kv, c, c, r, is_causal=True), attention_on_packed_rows(q, *kv, c, r, is_causal=True)):
        assert got[:, :, :key].isfinite().all() and not got[:, :, key:].isfinite().any()
        assert torch.equal(got.isfinite(), attention_in_one_piece(q, *kv, c, r, is_causal=True).isfinite())


def _rows_close(got, want, limit, what=""):
    """The worst row's relative error (2-norms over the last dimension)."""
    got, want = got.cpu().double().flatten(0, -2), want.cpu().double().flatten(0, -2)
    rel = (got - want).norm(dim=1) / want.norm(dim=1)
    assert rel.max() <= limit, f"{what} row {int(rel.argmax())}: relative error {rel.max():.2e}, limit {limit:.2e}"


@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("nq", [3, 12])
def test_rows_of_very_different_size_in_one_block(nq, d, paged):
    """Every other row attends to one token whose value is some 2^32 times the others': the rows beside it keep their precision
    (the combine launch rotates 4 or 16 rows at a time)."""
    hq, hkv, n, bs, dtype = 4, 1, 2111, 16, torch.bfloat16
    assert attention_workspace_bytes(1, nq, n, hq, hkv, d) > 0
    kv, c, r = _packed(1, hkv, n, d, 101)
    kv[3] *= 0.05
    kv[3][..., 0, :] = 1e9
    key = O.decompress(kv[0].reshape(1, n, d // 2), kv[1].reshape(1, n, 1), c)[0, 0] @ r          # the key of that token
    q = torch.randn(1, hq, nq, d, generator=torch.Generator().manual_seed(102)) * 0.5
    q += 60 * d ** 0.5 / 11.3 * (key / key.norm()) * torch.tensor([1.0, -1.0]).repeat(nq)[:nq, None]
    q = q.to(dtype)
    want = O.fused_tq_attention(q, *kv, c, c, r).float()          # (its rotated query is rounded as the kernel's is)
    assert want[0, :, 0].norm() > 2e8 * want[0, :, 1].norm()
    dev = [t.to(DEV) for t in (*kv, c, r)]
    if paged:
        pages = (n + bs - 1) // bs
        cache = torch.zeros(pages, bs, hkv * (d + 8), dtype=torch.uint8)
        O.store_rows(cache, torch.arange(n), kv[0][0].transpose(0, 1).contiguous(), kv[1][0].transpose(0, 1).contiguous(),
                     kv[2][0].transpose(0, 1).contiguous(), kv[3][0].transpose(0, 1).contiguous())
        args = (torch.tensor([0, nq], dtype=torch.int32, device=DEV), nq, cache.to(DEV),
                torch.arange(pages, dtype=torch.int32, device=DEV)[None], torch.tensor([n], dtype=torch.int32, device=DEV), dev[4])
        qd = q[0].transpose(0, 1).contiguous().to(DEV)
        got = K.paged_tq4_prefill(qd, *args, dev[4], dev[5], hkv, d, bs, causal=False).transpose(0, 1)[None]
        one = prefill_in_one_piece(qd, *args, dev[5], hkv, d, bs, causal=False).transpose(0, 1)[None]
    else:
        qd = q.to(DEV)
        got = K.fused_tq_attention(qd, *dev[:5], dev[4], dev[5])
        one = attention_in_one_piece(qd, *dev[:4], dev[4], dev[5])
    # a rounding to bf16 moves a row by less than 2^-9 of its norm: the result and the output here, the output there; weights
    # and keys are held in fp16 (2^-10 of a weight, and a key's 2^-12 moves a score of up to 60 by less than
    # 60 * 2^-12 / sqrt(d) < 2^-9)
    limit = 3 * 2 ** -9 + 2 ** -10 + 2 ** -9
    _rows_close(one, want, limit, "in one piece")
    _rows_close(got, want, limit, "in pieces")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("nq,n", [(2, 1), (2, 2111), (40, 2111), (400, 4100)])
def test_coordinates_of_very_different_size_in_one_row(nq, n, d, dtype):
    """Paged rows are rounded to the query dtype and rotated back: with the identity as the matrix every coordinate comes
    out as it was rounded, also one 2^-20 of the row's largest."""
    hq, hkv, bs = 4, 1, 16
    if nq == 400:
        hq, hkv = 32, 8                                     # the combine launch by workgroups
    g = torch.Generator().manual_seed(103)
    c = torch.cat([-2.0 ** -10 * (1 + torch.rand(8, generator=g)), 2.0 ** 10 * (1 + torch.rand(8, generator=g))])
    token = torch.randint(0, 256, (hkv, d // 2), dtype=torch.uint8, generator=g)
    pages = (n + bs - 1) // bs
    cache = torch.zeros(pages, bs, hkv * (d + 8), dtype=torch.uint8)
    same = token[None].expand(n, hkv, d // 2).contiguous()
    ones = torch.ones(n, hkv, 1)
    O.store_rows(cache, torch.arange(n), same, ones, same, ones)
    q = (torch.randn(nq, hq, d, generator=g) * 1e-3).to(dtype).to(DEV)
    eye = torch.eye(d, device=DEV)
    args = (q, torch.tensor([0, nq], dtype=torch.int32, device=DEV), nq, cache.to(DEV), torch.arange(pages, dtype=torch.int32, device=DEV)[None],
            torch.tensor([n], dtype=torch.int32, device=DEV), c.to(DEV))
    value = c[O.nibble_unpack(token).long()].double().repeat_interleave(hq // hkv, 0)      # (heads, D)
    # held as fp16 (2^-11), the weights' sum as theirs (2^-11), rounded to the query dtype once: nothing more for one key
    limit = 2 * 2 ** -11 + (2 ** -8 if dtype == torch.bfloat16 else 2 ** -11)
    for got in (K.paged_tq4_prefill(*args, c.to(DEV), eye, hkv, d, bs, causal=False), prefill_on_packed_rows(*args, eye, hkv, d, bs, causal=False)):
        err = ((got.cpu().double() - value) / value).abs().max()
        assert err <= limit, f"{err:.2e}, limit {limit:.2e}"


# more sequences than are ordered: single queries (the grid has a place for every sequence), the same with one long prompt
# (most places of such a grid would be empty: the sequences are counted), short prompts of one and two workgroups
MANY = {"single": [1] * 300, "one prompt": [1] * 150 + [700] + [1] * 139 + [0, 40] * 5, "prompts": [(s * 37) % 90 for s in range(330)]}


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("many", list(MANY))
def test_paged_prefill_of_many_sequences(many, d):
    """Every row of every sequence is written once; the entry that does not know the number of tokens hands out the same."""
    ql, hq, hkv, bs, dtype = MANY[many], 8, 2, 16, torch.bfloat16
    kv = [n + (s * 29) % 50 if s % 7 else n for s, n in enumerate(ql)]
    c, _, r = book(d)
    _, cache, table, sl = build_paged_case(kv, hq, hkv, d=d, bs=bs, seed=111, dtype=dtype)
    q = torch.randn(sum(ql), hq, d, generator=torch.Generator().manual_seed(112)).to(dtype)
    cu = torch.tensor([0] + list(torch.tensor(ql).cumsum(0)), dtype=torch.int32)
    want = O.paged_prefill(q, cu, cache, table, sl, c, c, r, hkv, d, bs)
    args = (q.to(DEV), cu.to(DEV), max(ql), cache.to(DEV), table.to(DEV), sl.to(DEV), c.to(DEV))
    got = torch.full_like(q, 7.0).to(DEV)
    K.paged_tq4_prefill(*args, c.to(DEV), r.to(DEV), hkv, d, bs, out=got)
    # three roundings to bf16 and fp16 keys, a worst row of some thousands: as in _close with the row's own norm
    _rows_close(got, want, 4 * 2 ** -8)
    assert torch.equal(prefill_in_one_piece(*args, r.to(DEV), hkv, d, bs), got)


# (queries, keys) per sequence under a block table of 4096 tokens, which allows pieces that the lengths may not be worth:
# prompts of one and of several workgroups, long and short contexts together, sequences without queries or keys
UNDER_WIDE = [([400] * 3, [400] * 3), ([200] * 3, [700, 200, 900]), ([40, 1, 300, 0, 5], [2000, 300, 300, 50, 1100]),
              ([1, 1, 17, 1], [200, 0, 430, 900]), ([700, 64], [700, 1500])]


@pytest.mark.parametrize("hq,hkv,d", [(16, 4, 64), (16, 4, 128), (8, 2, 256), (8, 8, 128)])
@pytest.mark.parametrize("batch", range(len(UNDER_WIDE)))
def test_paged_prefill_under_a_wide_table(batch, hq, hkv, d):
    ql, kv = UNDER_WIDE[batch]
    bs, dtype = 16, torch.bfloat16
    assert attention_workspace_bytes(len(ql), max(ql), 4096, hq, hkv, d) > 0
    c, _, r = book(d)
    _, cache, table, sl = build_paged_case(kv, hq, hkv, d=d, bs=bs, seed=121, dtype=dtype)
    q = torch.randn(sum(ql), hq, d, generator=torch.Generator().manual_seed(122)).to(dtype)
    cu = torch.tensor([0] + list(torch.tensor(ql).cumsum(0)), dtype=torch.int32)
    want = O.paged_prefill(q, cu, cache, table, sl, c, c, r, hkv, d, bs)
    wide = torch.randint(-3, 1 << 20, (len(ql), 256), dtype=torch.int32, generator=torch.Generator().manual_seed(123))
    wide[:, :table.shape[1]] = table
    args = (q.to(DEV), cu.to(DEV), max(ql), cache.to(DEV), wide.to(DEV), sl.to(DEV), c.to(DEV))
    out = K.paged_tq4_prefill(*args, c.to(DEV), r.to(DEV), hkv, d, bs, out=torch.full_like(q, 7.0).to(DEV))
    keyless = torch.cat([torch.full((n,), m == 0) for n, m in zip(ql, kv)])
    for got in (out, prefill_on_packed_rows(*args, r.to(DEV), hkv, d, bs)):
        assert (got.cpu()[keyless] == 0).all()
        _rows_close(got.cpu()[~keyless], want[~keyless], 4 * 2 ** -8)


def test_paged_attention_under_capture_with_other_lengths():
    """One captured call: the pieces follow from the lengths that each replay finds on the device."""
    hq, hkv, d, bs, dtype = 16, 4, 128, 16, torch.bfloat16
    kv, ql = [3000, 900, 2500, 60], [1, 40, 200, 5]
    c, _, r = book(d)
    _, cache, table, sl = build_paged_case(kv, hq, hkv, d=d, bs=bs, seed=131, dtype=dtype)
    q = torch.randn(sum(ql), hq, d, generator=torch.Generator().manual_seed(132)).to(dtype).to(DEV)
    cu = torch.tensor([0] + list(torch.tensor(ql).cumsum(0)), dtype=torch.int32).to(DEV)
    sl = sl.to(DEV)
    out = torch.zeros_like(q)
    args = (cu, max(ql), cache.to(DEV), table.to(DEV), sl, c.to(DEV), c.to(DEV), r.to(DEV), hkv, d, bs)
    K.paged_tq4_prefill(q, *args, out=out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        K.paged_tq4_prefill(q, *args, out=out)
    for lens in (kv, [200, 900, 200, 5], [3000, 40, 2400, 60], [1, 41, 201, 6], kv):
        sl.copy_(torch.tensor(lens, dtype=torch.int32))
        eager = K.paged_tq4_prefill(q, *args)
        out.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
        want = O.paged_prefill(q.cpu(), cu.cpu(), cache, table, sl.cpu(), c, c, r, hkv, d, bs)
        _rows_close(out, want, 4 * 2 ** -8)


# (queries, keys): contexts of one tile, of tile counts that halve and quarter evenly and not, all alike, one long among short
SEARCH = [([1, 2, 3], [1, 64, 63]), ([33] * 4, [64, 128, 256, 512]), ([20, 300, 1], [65, 321, 449]), ([40] * 9, [200] * 9),
          ([1] * 64 + [500], [1] * 64 + [1700])]


@pytest.mark.parametrize("hq,hkv,d", [(3, 1, 128), (8, 2, 64), (2, 1, 256)])
@pytest.mark.parametrize("batch", range(len(SEARCH)))
def test_every_row_once_at_the_edges_of_the_search(batch, hq, hkv, d):
    """Workgroups find their work by the tile counts; with fewer than eight units some of their wavefronts have none."""
    ql, kv = SEARCH[batch]
    bs, dtype = 16, torch.float16
    c, _, r = book(d)
    _, cache, table, sl = build_paged_case(kv, hq, hkv, d=d, bs=bs, seed=91, dtype=dtype)
    q = torch.randn(sum(ql), hq, d, generator=torch.Generator().manual_seed(92)).to(dtype)
    cu = torch.tensor([0] + list(torch.tensor(ql).cumsum(0)), dtype=torch.int32)
    want = O.paged_prefill(q, cu, cache, table, sl, c, c, r, hkv, d, bs)
    args = (q.to(DEV), cu.to(DEV), max(ql), cache.to(DEV), table.to(DEV), sl.to(DEV), c.to(DEV))
    got = K.paged_tq4_prefill(*args, c.to(DEV), r.to(DEV), hkv, d, bs, out=torch.full_like(q, 7.0).to(DEV))
    _close(got, want, dtype)
    _close(prefill_on_packed_rows(*args, r.to(DEV), hkv, d, bs, out=torch.full_like(q, 7.0).to(DEV)), want, dtype)
