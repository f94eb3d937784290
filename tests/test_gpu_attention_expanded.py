"""Attention over expanded keys and values (many queries that share their keys), contiguous and paged: edges of the 32-row units, of
the tiles and of the blocks of 32 tokens, numbers of heads and pairs that the workgroups and the XCDs do not divide, long norms, numbers
that are none, workgroups in pieces, every row of a mixed batch."""
from __future__ import annotations

import ctypes

import pytest
import torch

from flashquant_amd import kernels as K
from oracle import tq_oracle as O
from tests.gpu_util import (_entry, attention_in_one_piece, attention_on_packed_rows, attention_workspace_bytes, book, build_paged_case,
                            prefill_on_packed_rows)

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _expanded(b, hkv, hq, nq, nkv, d, causal):
    """Whether a call of these sizes asks for room for its keys and values as fp16 (in tiles of 64 tokens, 32 at 256)."""
    tile = 32 if d == 256 else 64
    keys = min(nq, nkv) if causal else nkv
    return attention_workspace_bytes(b, nq, nkv, hq, hkv, d, 1 if causal else 2) >= b * hkv * -(-keys // tile) * tile * d * 4


def _inputs(b, hq, hkv, nq, nkv, d, dtype, seed):
    c, bnd, r = book(d)
    g = torch.Generator().manual_seed(seed)
    kv = []
    for _ in range(2):
        p, m = O.compress(torch.randn(b * hkv * nkv, 1, d, generator=g), r, bnd)
        kv += [p.reshape(b, hkv, nkv, d // 2), m.reshape(b, hkv, nkv, 1)]
    return torch.randn(b, hq, nq, d, generator=g).to(dtype), kv, c, r


def _attend(q, kv, c, r, causal, dev=DEV):
    return K.fused_tq_attention(q.to(dev), *[t.to(dev) for t in kv], c.to(dev), c.to(dev), r.to(dev), is_causal=causal)


def _close(got, want, dtype):
    """2-norms: bf16 rounds the rotated query (the oracle alone), the output there and here, 2^-9 of the norm each; fp16 the
    same, and keys, values and weights are held in fp16 (2^-12, the weights towards zero 2^-11; centroids and result of a key or
    value each): (3 + 2 + 2 + 4)^(1/2) * 2^-12.  Doubled."""
    limit = 2 * (3 ** 0.5 * 2 ** -9 if dtype == torch.bfloat16 else 11 ** 0.5 * 2 ** -12)
    got, want = got.cpu().double(), want.double()
    rel = (got - want).norm() / want.norm()
    assert rel <= limit, f"relative error {rel:.2e}, limit {limit:.2e}"
    row = (got - want).norm(dim=-1) / want.norm(dim=-1)
    assert row.max() <= 4 * limit, f"worst row {row.max():.2e}, limit {4 * limit:.2e}"


# (batch, query heads, KV heads, queries, keys, causal): a last unit of one row and of 31, one more key than a tile and one fewer,
# 1, 3 and 5 query heads a KV head (units of a workgroup at different positions), pairs that are and are not a multiple of 8, fewer
# keys than queries and more, workgroups with wavefronts that have no unit, more workgroups than two a CU
SIZES = [(1, 8, 8, 129, 129, True), (2, 5, 1, 191, 191, True), (1, 32, 8, 160, 160, True), (3, 6, 2, 193, 130, True), (1, 4, 1, 257, 300, True),
         (1, 8, 2, 255, 255, False), (2, 8, 1, 131, 65, False), (1, 12, 4, 320, 33, False), (8, 16, 2, 300, 300, True), (5, 24, 8, 385, 385, True)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("b,hq,hkv,nq,nkv,causal", SIZES)
def test_rows_at_the_edges(b, hq, hkv, nq, nkv, causal, d, dtype):
    if d == 64:                                               # (fewer queries stay on the other kernel there)
        nq, nkv = nq + 192, nkv + 128
    assert _expanded(b, hkv, hq, nq, nkv, d, causal)
    q, kv, c, r = _inputs(b, hq, hkv, nq, nkv, d, dtype, 7 * nq + d)
    want = O.fused_tq_attention(q, *kv, c, c, r, is_causal=causal)
    got = _attend(q, kv, c, r, causal)
    _close(got, want, dtype)
    assert torch.equal(_attend(q, kv, c, r.t().contiguous().t(), causal), got)          # the matrix in the other layout
    assert torch.equal(_attend(q, kv, c, r, causal), got)


def _in_64_bits(q, kv, c, r):
    """Causal attention of rows (1, heads, n, d) over one KV head in float64, the query not rounded once it is rotated."""
    k, v = (c.double()[O.nibble_unpack(p[0, 0]).long()] * m[0, 0].double() @ r.double() for p, m in (kv[:2], kv[2:]))
    n, d = k.shape
    scores = (q.double() @ k.T / d ** 0.5).masked_fill(torch.ones(n, n, dtype=torch.bool).triu(1), -torch.inf)
    return scores.softmax(-1) @ v


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("at", [0, 31, 32, 63, 64, 140])
def test_long_norms_beside_ordinary_ones(at, d):
    """A key and a value whose rows would not fit fp16, in every place of a tile: the rows that see them and the others."""
    b, hq, hkv, n, key_norm = 1, 4, 1, 210, 3e5
    assert _expanded(b, hkv, hq, n, n, d, True)
    q, kv, c, r = _inputs(b, hq, hkv, n, n, d, torch.float16, 31 + at)
    kv[1][..., at, :] = key_norm
    kv[3][..., at, :] = 1e5
    q *= 2e-4
    want = _in_64_bits(q, kv, c, r)
    assert (want[:, :, at:].norm(dim=-1) > 1e3).double().mean() > 0.25 and want.abs().max() < 65504
    got = _attend(q, kv, c, r, True)
    if at:
        _close(got[:, :, :at], want[:, :, :at], torch.float16)
    # Rounding that key (centroids and result, 2^-12 of its norm each) moves its scores by at most `moved`, and with them its weight;
    # the value that it weighs is the most of the rows that see it.
    moved = 2 ** 0.5 * 2 ** -12 * q.double().norm(dim=-1).max() * key_norm / d ** 0.5
    err = (got.cpu().double() - want).norm(dim=-1) / want.norm(dim=-1)
    limit = moved + 8 * 11 ** 0.5 * 2 ** -12
    assert moved < 0.03 and err[:, :, at:].max() <= limit, f"worst row {err.max():.2e}, limit {limit:.2e}"


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("side", [1, 3])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_numbers_that_are_none_stay_visible(value, side, d):
    """Rows in front of such a key see nothing of it; the others are no numbers, as in the kernel that does not expand.  (A value's
    tile is multiplied as a whole: rows of the same 32 tokens in front of it may show it.)"""
    b, hq, hkv, n, at = 1, 8, 2, 400, 200
    assert _expanded(b, hkv, hq, n, n, d, True)
    q, kv, c, r = _inputs(b, hq, hkv, n, n, d, torch.bfloat16, 5)
    kv[side][:, 0, at] = value
    got = _attend(q, kv, c, r, True)
    one = attention_in_one_piece(q.to(DEV), *[t.to(DEV) for t in kv], c.to(DEV), r.to(DEV), is_causal=True)
    seen = at if side == 1 else at // 64 * 64
    assert got[:, :4, :seen].isfinite().all() and got[:, 4:].isfinite().all()
    assert not got[:, :4, at:].isfinite().any() and not one[:, :4, at:].isfinite().any()


def test_under_capture():
    b, hq, hkv, n, d = 2, 16, 4, 333, 128
    q, kv, c, r = _inputs(b, hq, hkv, n, n, d, torch.bfloat16, 17)
    dev = [t.to(DEV) for t in kv]
    q, c, r = q.to(DEV), c.to(DEV), r.to(DEV)
    K.fused_tq_attention(q, *dev, c, c, r, is_causal=True)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = K.fused_tq_attention(q, *dev, c, c, r, is_causal=True)
    for k in range(4):
        q.copy_(torch.randn(q.shape, generator=torch.Generator().manual_seed(63 + k)).to(q.dtype))
        eager = K.fused_tq_attention(q, *dev, c, c, r, is_causal=True)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)


def test_pairs_that_take_turns_in_the_workspace():
    """More images than the workspace holds at a time: 72 KV heads of 16,448 tokens, 63 of which fit."""
    b, h, n, d = 1, 72, 16448, 256
    assert h * n * d * 4 > 2 ** 30 and 0.9 * 2 ** 30 < attention_workspace_bytes(b, n, n, h, h, d, 1) < 1.1 * 2 ** 30
    c, _, r = (t.to(DEV) if isinstance(t, torch.Tensor) else t for t in book(d))
    g = torch.Generator(device=DEV).manual_seed(3)
    kv = []
    for _ in range(2):
        kv += [torch.randint(0, 256, (b, h, n, d // 2), dtype=torch.uint8, device=DEV, generator=g),
               d ** 0.5 * (0.5 + torch.rand(b, h, n, 1, device=DEV, generator=g))]
    q = torch.randn(b, h, n, d, device=DEV, generator=g).to(torch.bfloat16)
    got = K.fused_tq_attention(q, *kv, c, c, r, is_causal=True)
    want = attention_in_one_piece(q, *kv, c, r, is_causal=True)
    # bf16: query and output rounded there, the output here
    rel = ((got.float() - want.float()).flatten(2).norm(dim=2) / want.float().flatten(2).norm(dim=2)).max()
    assert rel <= 2 * 3 ** 0.5 * 2 ** -9, f"{rel:.2e}"


# (batch, query heads, KV heads, queries, keys, dimension, causal): prompts whose longest workgroups run in pieces (the last tile of one
# key, of all but one; rows that see nothing of a piece), and calls without a mask, whose workgroups all do
PIECES = [(1, 4, 1, 4033, 4033, 128, True), (1, 8, 1, 1535, 1535, 256, True), (2, 4, 1, 1601, 1601, 256, True), (1, 4, 1, 4033, 4033, 64, True),
          (1, 8, 1, 2033, 2305, 128, False), (1, 8, 1, 2033, 2497, 64, False), (1, 8, 1, 361, 655, 256, False)]


def _planned(b, hkv, hq, nq, nkv, d, causal):
    """Whether the workspace has room for the rows of pieces beside the images (4 rows of 32 and 64 numbers a slot)."""
    tile = 32 if d == 256 else 64
    tiles = b * hkv * -(-(min(nq, nkv) if causal else nkv) // tile)
    return attention_workspace_bytes(b, nq, nkv, hq, hkv, d, 1 if causal else 2) - tiles * tile * (4 * d + 16) > 500 * 16 * (32 * d + 64)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,hq,hkv,nq,nkv,d,causal", PIECES)
def test_prompts_in_pieces(b, hq, hkv, nq, nkv, d, causal, dtype):
    assert _planned(b, hkv, hq, nq, nkv, d, causal)
    q, kv, c, r = _inputs(b, hq, hkv, nq, nkv, d, dtype, nq + d)
    kv[1][:, :, 37] *= 4e3                                    # a tile with a long norm in one piece
    q *= 0.5
    want = O.fused_tq_attention(q, *kv, c, c, r, is_causal=causal)
    got = _attend(q, kv, c, r, causal)
    err = (got.cpu().double() - want.double()).norm() / want.double().norm()
    # (scores of that key reach 4e3 times the others': one weight is all or nothing there, and a rounded query moves it)
    assert err <= 8 * 3 ** 0.5 * 2 ** -9
    kv[1][:, :, 37] /= 4e3
    _close(_attend(q, kv, c, r, causal), O.fused_tq_attention(q, *kv, c, c, r, is_causal=causal), dtype)


def _paged_expanded(ql, kv_room, hq, hkv, d):
    f = _entry("fq_paged_prefill_workspace_bytes", ctypes.c_size_t)
    need = f(ctypes.c_int(len(ql)), ctypes.c_int(max(ql)), ctypes.c_int64(kv_room), ctypes.c_int64(sum(ql)), ctypes.c_int(hq),
             ctypes.c_int(hkv), ctypes.c_int(d))
    return need > attention_workspace_bytes(len(ql), max(ql), kv_room, hq, hkv, d)


# (queries, keys): prompts, chunks with keys in front, single queries, idle sequences and ones without keys; key counts at and around
# tiles; more sequences than a wavefront has lanes, and the most that the plan takes; long workgroups beside short ones
BATCHES = [([600, 1, 64, 0, 129, 5], [600, 700, 500, 90, 129, 0]), ([257], [1025]), ([64, 63, 65, 300], [64, 63, 65, 300]),
           ([260 + s % 5 for s in range(70)], [260 + s % 5 + 13 * (s % 7) for s in range(70)]), ([33 * (s % 17) for s in range(256)], [33 * (s % 17) + s % 3 for s in range(256)]),
           ([2001, 1, 40, 1], [2001, 1900, 1500, 3])]


# (batch, query heads, KV heads, dimension, tokens of a page, type): all in bf16 on pages of 16, many sequences at one dimension; fp16 and
# the other pages on the first
PAGED = [(i, *heads, 16, torch.bfloat16) for i in range(len(BATCHES)) for heads in ((8, 2, 128), (5, 1, 128), (16, 2, 64), (8, 1, 256), (6, 2, 256))
         if i != 4 or heads[2] == 128]
PAGED += [(0, *heads, bs, dtype) for heads in ((8, 2, 128), (16, 2, 64), (8, 1, 256))
          for bs, dtype in ((16, torch.float16), (8, torch.float16), (32, torch.float16), (8, torch.bfloat16), (32, torch.bfloat16))]


@pytest.mark.parametrize("batch,hq,hkv,d,bs,dtype", PAGED)
def test_every_row_of_a_paged_batch(batch, hq, hkv, d, bs, dtype):
    ql, kv = BATCHES[batch]
    if d == 64:                                               # (shorter prompts stay on the other kernel there)
        ql, kv = [4 * n for n in ql[:20]], kv[:20]
        kv = [n + m // 4 * 3 if n else 0 for n, m in zip(kv, ql)]
    c, _, r = book(d)
    _, cache, table, sl = build_paged_case(kv, hq, hkv, d=d, bs=bs, seed=141, dtype=dtype)
    q = torch.randn(sum(ql), hq, d, generator=torch.Generator().manual_seed(142)).to(dtype)
    cu = torch.tensor([0] + list(torch.tensor(ql).cumsum(0)), dtype=torch.int32)
    assert _paged_expanded(ql, table.shape[1] * bs, hq, hkv, d)
    room = torch.randint(-3, 1 << 20, table.shape, dtype=torch.int32, generator=torch.Generator().manual_seed(143))
    pages = (torch.tensor(kv) + bs - 1) // bs
    dirty = torch.where(torch.arange(table.shape[1])[None] < pages[:, None], table, room)      # ids past a sequence's pages
    for causal in (True, False):
        want = O.paged_prefill(q, cu, cache, table, sl, c, c, r, hkv, d, bs, causal=causal)
        out = torch.full((q.numel() + 8,), 7.0, dtype=dtype, device=DEV)
        got = out[1:1 + q.numel()].view_as(q)                                                  # not 16-byte aligned
        K.paged_tq4_prefill(q.to(DEV), cu.to(DEV), max(ql), cache.to(DEV), dirty.to(DEV), sl.to(DEV), c.to(DEV), c.to(DEV), r.to(DEV),
                            hkv, d, bs, causal=causal, out=got)
        assert (out[:1] == 7).all() and (out[1 + q.numel():] == 7).all()
        keyless = torch.cat([torch.full((n,), m == 0) for n, m in zip(ql, kv)])
        assert (got.cpu()[keyless] == 0).all()
        rel = (got.cpu().float() - want.float()).norm(dim=-1) / want.float().norm(dim=-1)
        # bf16: query, result and output rounded there, the output here; fp16: as in _close; a worst row of some thousands
        limit = 2 * 2 * 2 ** -9 if dtype == torch.bfloat16 else 2 * 11 ** 0.5 * 2 ** -12
        assert rel[~keyless].max() <= (4 * 2 ** -8 if dtype == torch.bfloat16 else 4 * limit)
        assert rel[~keyless].square().mean().sqrt() <= limit
        assert torch.equal(K.paged_tq4_prefill(q.to(DEV), cu.to(DEV), max(ql), cache.to(DEV), table.to(DEV), sl.to(DEV), c.to(DEV), c.to(DEV),
                                               r.to(DEV), hkv, d, bs, causal=causal), got)


def test_paged_under_capture_with_other_lengths():
    """One captured call: the plan follows from the lengths that each replay finds on the device."""
    hq, hkv, d, bs, dtype = 16, 4, 128, 16, torch.bfloat16
    kv, ql = [900, 700, 1200, 60], [300, 40, 600, 5]
    c, _, r = book(d)
    _, cache, table, sl = build_paged_case(kv, hq, hkv, d=d, bs=bs, seed=151, dtype=dtype)
    assert _paged_expanded(ql, table.shape[1] * bs, hq, hkv, d)
    q = torch.randn(sum(ql), hq, d, generator=torch.Generator().manual_seed(152)).to(dtype).to(DEV)
    cu = torch.tensor([0] + list(torch.tensor(ql).cumsum(0)), dtype=torch.int32).to(DEV)
    sl = sl.to(DEV)
    out = torch.zeros_like(q)
    args = (cu, max(ql), cache.to(DEV), table.to(DEV), sl, c.to(DEV), c.to(DEV), r.to(DEV), hkv, d, bs)
    K.paged_tq4_prefill(q, *args, out=out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        K.paged_tq4_prefill(q, *args, out=out)
    for lens in (kv, [300, 700, 600, 5], [900, 40, 1199, 60], [301, 41, 601, 6], kv):
        sl.copy_(torch.tensor(lens, dtype=torch.int32))
        eager = K.paged_tq4_prefill(q, *args)
        out.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
        want = O.paged_prefill(q.cpu(), cu.cpu(), cache, table, sl.cpu(), c, c, r, hkv, d, bs)
        rel = (out.cpu().float() - want.float()).norm(dim=-1) / want.float().norm(dim=-1)
        assert rel.max() <= 4 * 2 ** -8


class _LittleMemory:
    """At most `spare` bytes more than what torch's allocator holds now (and nothing larger in what it holds)."""

    def __init__(self, spare):
        self.spare = spare

    def __enter__(self):
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        total = torch.cuda.get_device_properties(0).total_memory
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + self.spare) / total)

    def __exit__(self, *exc):
        torch.cuda.set_per_process_memory_fraction(1.0)


def _random_rows(b, h, n, d, g):
    return [t for _ in range(2) for t in (torch.randint(0, 256, (b, h, n, d // 2), dtype=torch.uint8, device=DEV, generator=g),
                                          d ** 0.5 * (0.5 + torch.rand(b, h, n, 1, device=DEV, generator=g)))]


@pytest.mark.parametrize("causal", [True, False])
def test_without_room_for_expanded_keys(causal):
    """A call whose expanded keys (96 MiB) do not fit the memory that is left runs on the packed ones."""
    b, h, n, d = 1, 32, 6144, 128
    assert _expanded(b, h, h, n, n, d, causal)
    c, _, r = (t.to(DEV) for t in book(d))
    g = torch.Generator(device=DEV).manual_seed(7)
    kv = _random_rows(b, h, n, d, g)
    q = torch.randn(b, h, n, d, device=DEV, generator=g, dtype=torch.bfloat16)
    want = attention_on_packed_rows(q, *kv, c, r, is_causal=causal).cpu()
    with _LittleMemory(90 << 20):                              # (the result takes 48 MiB, rows of pieces 33)
        got = K.fused_tq_attention(q, *kv, c, c, r, is_causal=causal)
    assert torch.equal(got.cpu(), want)
    roomy = K.fused_tq_attention(q, *kv, c, c, r, is_causal=causal).cpu()
    assert not torch.equal(roomy, want)
    rel = (roomy.float() - want.float()).norm() / want.float().norm()
    assert rel <= 2 * 3 ** 0.5 * 2 ** -9                       # bf16: query and output rounded there, the output here


def test_paged_without_room_for_expanded_keys():
    ql, kv, hq, hkv, d, bs = [2000, 1500, 1], [2000, 1900, 700], 16, 16, 128, 16
    c, _, r = (t.to(DEV) for t in book(d))
    g = torch.Generator(device=DEV).manual_seed(8)
    pages = 3 * 125
    assert _paged_expanded(ql, 125 * bs, hq, hkv, d)
    cache = torch.randint(0, 256, (pages, bs, hkv * (d + 8)), dtype=torch.uint8, device=DEV, generator=g)
    norms = cache.view(-1, hkv * (d + 8)).view(torch.float32)
    norms[:, hkv * 16:hkv * 17] = d ** 0.5 * (0.5 + torch.rand(pages * bs, hkv, device=DEV, generator=g))
    norms[:, hkv * 33:] = d ** 0.5 * (0.5 + torch.rand(pages * bs, hkv, device=DEV, generator=g))
    table = torch.randperm(pages, device=DEV, generator=g).to(torch.int32).view(3, 125)
    q = torch.randn(sum(ql), hq, d, device=DEV, generator=g, dtype=torch.bfloat16)
    cu = torch.tensor([0] + list(torch.tensor(ql).cumsum(0)), dtype=torch.int32, device=DEV)
    args = (cu, max(ql), cache, table, torch.tensor(kv, dtype=torch.int32, device=DEV), c)
    want = prefill_on_packed_rows(q, *args, r, hkv, d, bs).cpu()
    torch.cuda.empty_cache()
    out = torch.empty_like(q)
    with _LittleMemory(40 << 20):
        K.paged_tq4_prefill(q, *args, c, r, hkv, d, bs, out=out)
    assert torch.equal(out.cpu(), want)
    assert not torch.equal(K.paged_tq4_prefill(q, *args, c, r, hkv, d, bs).cpu(), want)
