"""Performance cases of the TQ4 KV-cache path, through the entry points a serving program calls.

Each case is a dict of plain values; its ``kind`` names what a program does:

  step        one generated token per sequence in a serving loop: ``TQ4AttentionKernels.decode_step``
              (the new token's K and V into the paged cache, then attention over the context)
  decode      attention of one query per sequence over a filled cache: ``kernels.split_k_paged_decode``
  serve       a prefill batch of a serving loop: ``compress_and_store`` then ``prefill`` (fresh prompts,
              later chunks of long prompts and single-token queries mixed)
  attend      a whole prompt over contiguous packed keys and values: ``kernels.fused_tq_attention``, causal
  ring        a generated token of a model whose cache is a ring buffer: ``CompressedKVLayer.attend``
  compress    many rows to packed form: ``kernels.tq4_compress``
  materialise the paged cache back to 16-bit keys and values: ``TQ4AttentionKernels.decompress_cache``
  prod_step   one generated token per sequence over 3-bit + sign keys: ``prod_compress``, ``tq4_compress``,
              ``prod_store_rows``, ``prod_paged_decode``

Packed inputs are made with torch alone (indices of Gaussian coordinates, norms around sqrt(d)), so they do
not depend on the kernels that are measured.  Ragged lengths come from the case's own ``mix`` number.
"""
from __future__ import annotations

import math
import random

import torch

from flashquant_amd import kernels as K
from flashquant_amd import load_native
from flashquant_amd.cache import CompressedKVLayer
from flashquant_amd.kernels.prod import sketch_in_rotated_space
from flashquant_amd.vllm.impl import TQ4AttentionKernels

DEV = "cuda"
TYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    return [
        # one user on an 8-KV-head model of dimension 128, short context: launches and latency
        dict(name="step_1x777", kind="step", seqs=1, lo=777, hi=777, hq=32, hkv=8, d=128, page=16, type="bf16", mix=1),
        # the headline: a batch of 32 at 4096 tokens, as a serving loop runs it
        dict(name="step_32x4096", kind="step", seqs=32, lo=4096, hi=4096, hq=32, hkv=8, d=128, page=16, type="bf16", mix=1),
        # a larger ragged batch over long contexts, fp16 queries, 8 query heads per KV head
        dict(name="decode_61_ragged", kind="decode", seqs=61, lo=500, hi=16000, hq=64, hkv=8, d=128, page=16, type="fp16",
             mix=3),
        # one rank of eight of the same model under tensor parallelism: one KV head
        dict(name="step_96_shard", kind="step", seqs=96, lo=1000, hi=7000, hq=8, hkv=1, d=128, page=16, type="bf16", mix=4),
        # a small model with heads of 64
        dict(name="step_24_d64", kind="step", seqs=24, lo=200, hi=4000, hq=32, hkv=8, d=64, page=16, type="fp16", mix=5),
        # a scheduler's mixed batch: prompts, later chunks of prompts and generated tokens
        dict(name="serve_mixed", kind="serve", seqs=12, chunk=2048, hi=6000, hq=32, hkv=8, d=128, page=16, type="bf16",
             mix=6),
        # whole prompts of 8192 tokens over contiguous keys and values
        dict(name="attend_4x8192", kind="attend", batch=4, n=8192, hq=32, hkv=8, d=128, type="bf16"),
        # a prompt of a model with heads of 256
        dict(name="attend_3001_d256", kind="attend", batch=1, n=3001, hq=16, hkv=4, d=256, type="fp16"),
        # token by token generation on the ring-buffer cache
        dict(name="ring_4x2500", kind="ring", batch=4, n=2500, cap=4096, nq=1, hq=32, hkv=8, d=128, type="bf16"),
        # a large prompt set packed in one go (2,097,152 tokens of 8 heads)
        dict(name="compress_2M", kind="compress", n=2097152, h=8, d=128, type="bf16"),
        # the cache of a few thousand tokens back to keys and values in the original space
        dict(name="materialise_1501", kind="materialise", pages=1501, page=16, h=8, d=128, type="bf16", rotate=True),
        # long contexts on the 3-bit + sign record
        dict(name="prod_step_8", kind="prod_step", seqs=8, lo=16384, hi=131072, hq=64, hkv=8, page=16, type="bf16", mix=12),
    ]


# (query heads, KV heads, dimension): whole models and their tensor-parallel shards
HEADS = ((32, 8, 128), (64, 8, 128), (32, 4, 128), (16, 2, 128), (8, 1, 128), (32, 32, 128), (32, 8, 64), (16, 4, 64),
         (32, 8, 256), (16, 4, 256), (8, 1, 256))
MAX_CACHE = 600 << 20          # bytes of cache behind one drawn decode or step
MAX_FLOPS = 1.5e12             # of one drawn prefill


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("step", "step", "decode", "serve", "attend", "ring", "compress", "materialise", "prod_step"))
    ty = rng.choice(("bf16", "bf16", "fp16"))
    page = rng.choice((16, 16, 32))
    hq, hkv, d = rng.choice(HEADS)
    mix = rng.randrange(1, 1 << 20)
    if kind in ("step", "decode"):
        hi = _log(rng, 64, 32768)
        seqs = _log(rng, 1, min(256, max(1, MAX_CACHE // (hi * hkv * (d + 8)))))
        return dict(kind=kind, seqs=seqs, lo=max(1, hi // rng.choice((1, 4, 20))), hi=hi, hq=hq, hkv=hkv, d=d, page=page,
                    type=ty, mix=mix)
    if kind == "serve":
        chunk = _log(rng, 64, 4096)
        hi = chunk + _log(rng, 1, 8192)
        while True:
            seqs = _log(rng, 1, 24)
            case = dict(kind=kind, seqs=seqs, chunk=chunk, hi=hi, hq=hq, hkv=hkv, d=d, page=page, type=ty, mix=mix)
            if work(case)["flops"] <= MAX_FLOPS / (3 if d == 256 else 1):
                return case
            chunk, hi = max(64, chunk * 3 // 4), max(65, hi * 3 // 4)
    if kind == "attend":
        most = MAX_FLOPS / (3 if d == 256 else 1) / (2.0 * d * hq)
        n = _log(rng, 65, min(8192, int(math.sqrt(most))))
        batch = _log(rng, 1, max(1, min(8, int(most / (n * n)))))
        return dict(kind=kind, batch=batch, n=n, hq=hq, hkv=hkv, d=d, type=ty)
    if kind == "ring":
        n = _log(rng, 64, 16384)
        batch = _log(rng, 1, max(1, min(16, MAX_CACHE // (2 * n * hkv * (d + 8)))))
        return dict(kind=kind, batch=batch, n=n, cap=n + rng.randrange(1, 2048), nq=rng.choice((1, 1, 1, 2, 5)),
                    hq=hq, hkv=hkv, d=d, type=ty)
    if kind == "compress":
        return dict(kind=kind, n=_log(rng, 16, 1 << 20) * 8 // hkv * 128 // d, h=hkv, d=d, type=ty)
    if kind == "materialise":
        return dict(kind=kind, pages=_log(rng, 16, 8192) * 8 // hkv * 128 // d, page=page, h=hkv, d=d, type=ty,
                    rotate=rng.choice((True, True, False)))
    hi = _log(rng, 1024, 131072)
    seqs = _log(rng, 1, min(64, max(1, (480 << 20) // (hi * 1120))))
    return dict(kind=kind, seqs=seqs, lo=max(1, hi // rng.choice((1, 2, 8))), hi=hi, hq=rng.choice((32, 64)), hkv=8,
                page=page, type=ty, mix=mix)


# ---- sizes ------------------------------------------------------------------------------------------------

def _lens(case):
    r = random.Random(case["mix"])
    return [r.randint(case["lo"], case["hi"]) for _ in range(case["seqs"])]


def _serve_lens(case):
    """(new tokens, context including them) per sequence: half fresh prompts, a quarter later chunks, a quarter decodes."""
    r = random.Random(case["mix"])
    out = []
    for s in range(case["seqs"]):
        if s % 4 == 3:
            out.append((1, r.randint(2, case["hi"])))
        elif s % 4 == 1:
            new = r.randint(1, case["chunk"])
            out.append((new, new + r.randint(1, max(1, case["hi"] - case["chunk"]))))
        else:
            new = r.randint(max(1, case["chunk"] // 8), case["chunk"])
            out.append((new, new))
    return out


def work(case):
    k = case["kind"]
    d = case.get("d", 128)
    if k in ("step", "decode"):
        tokens, s, hq, hkv = sum(_lens(case)), case["seqs"], case["hq"], case["hkv"]
        extra = s * hkv * (4 * d + d + 8) if k == "step" else 0
        return {"bytes": tokens * hkv * (d + 8) + 4 * s * hq * d + extra, "flops": 4.0 * tokens * hq * d}
    if k == "prod_step":
        tokens, s, hq, hkv = sum(_lens(case)), case["seqs"], case["hq"], case["hkv"]
        return {"bytes": tokens * hkv * 140 + 4 * s * hq * d + s * hkv * (512 + 140), "flops": 6.0 * tokens * hq * d}
    if k == "serve":
        hq, hkv = case["hq"], case["hkv"]
        pairs = _serve_lens(case)
        new, ctx = sum(n for n, _ in pairs), sum(c for _, c in pairs)
        scores = sum(n * c - n * (n - 1) // 2 for n, c in pairs)
        return {"bytes": ctx * hkv * (d + 8) + 4 * new * hq * d + 4 * new * hkv * d + new * hkv * (d + 8),
                "flops": 4.0 * scores * hq * d}
    if k == "attend":
        b, n, hq, hkv = case["batch"], case["n"], case["hq"], case["hkv"]
        return {"bytes": b * n * (hkv * (d + 8) + 4 * hq * d), "flops": 2.0 * b * hq * d * n * (n + 1)}
    if k == "ring":
        b, n, hq, hkv = case["batch"], case["n"], case["hq"], case["hkv"]
        return {"bytes": b * n * hkv * (d + 8) + 4 * b * hq * case["nq"] * d, "flops": 4.0 * b * hq * case["nq"] * n * d}
    if k == "compress":
        rows = case["n"] * case["h"]
        return {"bytes": rows * (2 * d + d // 2 + 4), "flops": 2.0 * rows * d * d}
    rows = 2 * case["pages"] * case["page"] * case["h"]
    return {"bytes": rows * (2 * d + d // 2 + 4), "flops": 2.0 * rows * d * d if case["rotate"] else 1.0 * rows * d}


def tolerance(case):
    """About four times what two kernels of the library differ by on the same inputs (attention: its independent
    kernel variants, 2e-3 in bf16 and 5e-4 to 1e-3 in fp16; stored indices: the two- and the three-term rotation, 1.5e-5 of
    the bytes, or one or two bytes where few are stored; norms 1e-7)."""
    kind, bf16 = case["kind"], case["type"] == "bf16"
    if kind == "materialise":
        if not case["rotate"]:
            return "exact"                                   # one product and two roundings, in a given order
        return {"rel": 2e-3, "max": 2e-2} if bf16 else {"rel": 3e-4, "max": 4e-3}
    tol = {"rel": 8e-3, "max": 0.15} if bf16 else {"rel": 3e-3, "max": 0.05}
    if kind == "compress":
        tol = {"rel": 4e-7, "max": 1e-6}
        stored = case["n"] * case["h"] * case["d"] // 2
    elif kind in ("step", "serve", "prod_step"):
        tokens = sum(c for _, c in _serve_lens(case)) if kind == "serve" else sum(_lens(case))
        stored = tokens * case["hkv"] * case.get("d", 128) // 2
    else:
        return tol
    if kind == "serve":
        tol["max"] = 0.9          # the first tokens of a prompt attend to a few rows: one index at a tie shows there
    return {**tol, "differ": min(0.01, 6e-5 + 2.0 / stored)}


# ---- inputs -----------------------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, dtype):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32).to(dtype)


def _outlier_rows(g, n, h, d, dtype):
    """N(0, 1) rows with 4 channels of every head ten times larger, as keys of trained models have."""
    gain = torch.ones(h, d, device=DEV)
    gain.scatter_(1, torch.rand(h, d, generator=g, device=DEV).topk(4, dim=1).indices, 10.0)
    x = torch.empty(n, h, d, dtype=dtype, device=DEV)
    for part in x.split(max(1, (1 << 27) // (h * d))):
        part.copy_(torch.randn(part.shape, generator=g, device=DEV) * gain)
    return x


def _packed(g, rows, d, boundaries, bits=4):
    """(nibble-packed indices (rows, d / 2), norms (rows,)) of rows with Gaussian coordinates."""
    packed = torch.empty(rows, d // 2, dtype=torch.uint8, device=DEV)
    for part in packed.split(max(1, (1 << 26) // d)):
        y = torch.randn(part.shape[0], d, generator=g, device=DEV) / math.sqrt(d)
        idx = torch.bucketize(y, boundaries, out_int32=True).to(torch.uint8)
        if bits == 3:                                        # the sign of the sketched residual in bit 3
            idx |= torch.randint(0, 2, idx.shape, generator=g, device=DEV, dtype=torch.uint8) << 3
        part.copy_(idx[:, 0::2] << 4 | idx[:, 1::2])
    norms = math.sqrt(d) * torch.exp(0.25 * torch.randn(rows, generator=g, device=DEV))
    return packed, norms


def _tables(seed, lens, page):
    pages = [(n + page - 1) // page for n in lens]
    perm = torch.randperm(sum(pages), generator=torch.Generator().manual_seed(int(seed))).to(torch.int32)
    table = torch.zeros(len(lens), max(pages), dtype=torch.int32)
    first = 0
    for s, n in enumerate(pages):
        table[s, :n] = perm[first:first + n]
        first += n
    return table, sum(pages)


def _slots(table, page, s, start, end):
    t = torch.arange(start, end)
    return table[s].long()[t // page] * page + t % page


def _sections(cache, h, d):
    """The cache as what it holds: index bytes and norms of keys and of values (views)."""
    row = cache.view(-1, cache.shape[-1])
    o1, o2 = h * d // 2, h * d // 2 + 4 * h
    o3 = o2 + h * d // 2
    return {"k_index": row[:, :o1], "k_norm": row[:, o1:o2].view(torch.float32), "v_index": row[:, o2:o3],
            "v_norm": row[:, o3:].view(torch.float32)}


def _fill(g, cache, h, d, boundaries):
    for part in cache.view(-1, cache.shape[-1]).split(max(1, (1 << 20) // h)):
        sec = _sections(part, h, d)
        for side in "kv":
            p, n = _packed(g, part.shape[0] * h, d, boundaries)
            sec[side + "_index"].copy_(p.view(part.shape[0], -1))
            sec[side + "_norm"].copy_(n.view(part.shape[0], -1))


def _book(d, bits=4):
    centroids, boundaries = load_native().codebook.solve_lloyd_max(d, bits)
    return centroids.to(DEV), boundaries.to(DEV)


def prepare(case, seed):
    kind, g = case["kind"], _gen(seed)
    d, ty = case.get("d", 128), TYPES[case["type"]]
    st = {"kind": kind, "case": case}
    if kind in ("step", "decode", "serve"):
        hq, h, page = case["hq"], case["hkv"], case["page"]
        layer = TQ4AttentionKernels(h, d, 1.0 / math.sqrt(d), torch.device(DEV))
        pairs = _serve_lens(case) if kind == "serve" else [(1, n) for n in _lens(case)]
        lens = [c for _, c in pairs]
        table, pages = _tables(seed, lens, page)
        cache = torch.empty(pages, page, h * (d + 8), dtype=torch.uint8, device=DEV)
        _fill(g, cache, h, d, layer.boundaries)
        new = sum(n for n, _ in pairs)
        slots = torch.cat([_slots(table, page, s, c - n, c) for s, (n, c) in enumerate(pairs)])
        cu = torch.tensor([0] + [n for n, _ in pairs]).cumsum(0).to(torch.int32)
        q = _randn(g, new, hq, d, dtype=ty)
        st.update(layer=layer, cache=cache, sections=_sections(cache, h, d), table=table.to(DEV), slots=slots.to(DEV),
                  lens=torch.tensor(lens, dtype=torch.int32, device=DEV), cu=cu.to(DEV), most=max(n for n, _ in pairs),
                  q=q, out=torch.zeros_like(q), k=_outlier_rows(g, new, h, d, ty), v=_randn(g, new, h, d, dtype=ty))
    elif kind == "prod_step":
        hq, h, page, lens = case["hq"], case["hkv"], case["page"], _lens(case)
        native = load_native()
        st["rotation"], st["sketch"] = native.haar_orthogonal(d, 42).to(DEV), native.qjl_matrix(d, 42).to(DEV)
        st["sketch_rot"] = sketch_in_rotated_space(st["sketch"], st["rotation"])
        st["even"], st["odd"] = (t.to(DEV) for t in native.split_rotation(native.haar_orthogonal(d, 42)))
        st["c3"], st["b3"] = _book(d, 3)
        st["c4"], st["b4"] = _book(d)
        table, pages = _tables(seed, lens, page)
        kn, kg, vi, vn, row_bytes = K.prod_page_layout(h, d)
        cache = torch.empty(pages, page, row_bytes, dtype=torch.uint8, device=DEV)

        def sections(rows):
            return {"k_index": rows[:, :kn], "k_norm": rows[:, kn:kg].view(torch.float32),
                    "k_residual": rows[:, kg:vi].view(torch.float32), "v_index": rows[:, vi:vn],
                    "v_norm": rows[:, vn:].view(torch.float32)}

        for part in cache.view(-1, row_bytes).split((1 << 20) // h):
            sec, n = sections(part), part.shape[0]
            p, norm = _packed(g, n * h, d, st["b3"], bits=3)
            sec["k_index"].copy_(p.view(n, -1))
            sec["k_norm"].copy_(norm.view(n, -1))
            sec["k_residual"].copy_(norm.view(n, -1) * 0.185)      # what a 3-bit codebook leaves of a Gaussian row
            p, norm = _packed(g, n * h, d, st["b4"])
            sec["v_index"].copy_(p.view(n, -1))
            sec["v_norm"].copy_(norm.view(n, -1))
        slots = torch.cat([_slots(table, page, s, n - 1, n) for s, n in enumerate(lens)])
        q = _randn(g, len(lens), hq, d, dtype=ty)
        st.update(cache=cache, sections=sections(cache.view(-1, row_bytes)), table=table.to(DEV), slots=slots.to(DEV),
                  lens=torch.tensor(lens, dtype=torch.int32, device=DEV), q=q, out=torch.zeros_like(q),
                  k=_outlier_rows(g, len(lens), h, d, ty), v=_randn(g, len(lens), h, d, dtype=ty))
    elif kind in ("attend", "ring"):
        b, n, hq, h = case["batch"], case["n"], case["hq"], case["hkv"]
        rotation = load_native().haar_orthogonal(d, 42)
        cent, bnd = _book(d)
        kv = []
        for _ in range(2):
            p, norm = _packed(g, b * h * n, d, bnd)
            kv += [p.view(b, h, n, d // 2), norm.view(b, h, n, 1)]
        if kind == "attend":
            st.update(q=_randn(g, b, hq, n, d, dtype=ty), kv=kv, rotation=rotation.to(DEV), centroids=cent)
        else:
            ring = CompressedKVLayer(case["cap"], b, h, d, rotation, cent, bnd)
            ring.keys.append(kv[0], kv[1])
            ring.values.append(kv[2], kv[3])
            st.update(q=_randn(g, b, hq, case["nq"], d, dtype=ty), ring=ring)
    elif kind == "compress":
        n, h = case["n"], case["h"]
        native = load_native()
        rotation = native.haar_orthogonal(d, 42)
        st["rotation"], (st["even"], st["odd"]) = rotation.to(DEV), (t.to(DEV) for t in native.split_rotation(rotation))
        st.update(x=_outlier_rows(g, n, h, d, ty), boundaries=_book(d)[1],
                  out=(torch.empty(n, h, d // 2, dtype=torch.uint8, device=DEV), torch.empty(n, h, 1, device=DEV)))
    else:
        h = case["h"]
        layer = TQ4AttentionKernels(h, d, 1.0 / math.sqrt(d), torch.device(DEV))
        cache = torch.empty(case["pages"], case["page"], h * (d + 8), dtype=torch.uint8, device=DEV)
        _fill(g, cache, h, d, layer.boundaries)
        st.update(layer=layer, cache=cache, type=ty, rotate=case["rotate"])
    return st


# ---- one pass ---------------------------------------------------------------------------------------------

def run(st):
    kind = st["kind"]
    if kind == "step":
        out = st["layer"].decode_step(st["q"], st["k"], st["v"], st["cache"], st["slots"], st["table"], st["lens"],
                                      out=st["out"])
        return {"out": out, **st["sections"]}
    if kind == "decode":
        y = st["layer"]
        return K.split_k_paged_decode(st["q"], st["cache"], st["table"], st["lens"], y.centroids, y.centroids, y.rotation,
                                      y.num_kv_heads, y.head_size, st["cache"].shape[1], sm_scale=y.scale, out=st["out"])
    if kind == "serve":
        st["layer"].compress_and_store(st["k"], st["v"], st["cache"], st["slots"])
        out = st["layer"].prefill(st["q"], st["cu"], st["most"], st["cache"], st["table"], st["lens"], out=st["out"])
        return {"out": out, **st["sections"]}
    if kind == "attend":
        return K.fused_tq_attention(st["q"], *st["kv"], st["centroids"], st["centroids"], st["rotation"], is_causal=True)
    if kind == "ring":
        return st["ring"].attend(st["q"])
    if kind == "compress":
        return K.tq4_compress(st["x"], st["rotation"], st["boundaries"], rotation_T_even=st["even"],
                              rotation_T_odd=st["odd"], out=st["out"])
    if kind == "materialise":
        return st["layer"].decompress_cache(st["cache"], st["type"], apply_rotation=st["rotate"])
    h, d = st["k"].shape[1:]
    kp, kn, kg = K.prod_compress(st["k"], st["rotation"], st["sketch"], st["b3"], st["c3"], sketch_rot=st["sketch_rot"])
    vp, vn = K.tq4_compress(st["v"], st["rotation"], st["b4"], rotation_T_even=st["even"], rotation_T_odd=st["odd"])
    K.prod_store_rows(st["cache"], st["slots"], kp, kn, kg, vp, vn)
    out = K.prod_paged_decode(st["q"], st["cache"], st["table"], st["lens"], st["c3"], st["c4"], st["rotation"],
                              st["sketch"], h, d, st["cache"].shape[1], out=st["out"])
    return {"out": out, **st["sections"]}
