"""Helpers for the GPU parity tests: seeded inputs, oracle-built paged caches."""
from __future__ import annotations

import ctypes
import os

import torch

from oracle import tq_oracle as O

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flashquant_amd", "libfq_hip.so")

_BOOKS = {}


def book(dim=128, bits=4, seed=42):
    key = (dim, bits, seed)
    if key not in _BOOKS:
        c, b = O.lloyd_max_gaussian(dim, bits)
        _BOOKS[key] = (c, b, O.haar_orthogonal(dim, seed))
    return _BOOKS[key]


def build_paged_case(lens, hq, hkv, d=128, bs=16, seed=3, dtype=torch.bfloat16, extra_blocks=3,
                     kv_scale=1.0):
    """Random K/V per sequence, compressed by the oracle and scattered into a
    paged cache through a seeded random block table.  Unused slots hold random
    bytes, so reads past a sequence's end would show up in the result."""
    c, b, r = book(d)
    g = torch.Generator().manual_seed(seed)
    S = len(lens)
    max_blocks = max(1, (max(lens) + bs - 1) // bs)
    nb = S * max_blocks + extra_blocks
    row = hkv * (d + 8)
    cache = torch.randint(0, 256, (nb, bs, row), dtype=torch.uint8, generator=g)
    # random bytes in the norm slots could decode to NaN/Inf; such slots are never
    # read by a correct kernel, and a wrong read then fails loudly
    table = torch.randperm(nb, generator=g)[: S * max_blocks].reshape(S, max_blocks).int()
    for s, L in enumerate(lens):
        if L == 0:
            continue
        k = torch.randn(L, hkv, d, generator=g) * kv_scale
        v = torch.randn(L, hkv, d, generator=g) * kv_scale
        kp, kn = O.compress(k, r, b)
        vp, vn = O.compress(v, r, b)
        t = torch.arange(L)
        slots = table[s].long()[t // bs] * bs + t % bs
        O.store_rows(cache, slots, kp, kn, vp, vn)
    q = torch.randn(S, hq, d, generator=g).to(dtype)
    return q, cache, table, torch.tensor(lens, dtype=torch.int32)


def _entry(name, restype=ctypes.c_int):
    f = getattr(ctypes.CDLL(LIB), name)
    f.restype = restype
    return f


def _args(*values):
    """Tensors as their addresses, ints as 64-bit or 32-bit C integers (None: NULL, (n,): int64)."""
    out = []
    for v in values:
        if v is None:
            out.append(ctypes.c_void_p(0))
        elif isinstance(v, torch.Tensor):
            assert v.is_contiguous()
            out.append(ctypes.c_void_p(v.data_ptr()))
        elif isinstance(v, tuple):
            out.append(ctypes.c_int64(v[0]))
        elif isinstance(v, float):
            out.append(ctypes.c_float(v))
        else:
            out.append(ctypes.c_int(v))
    return out


def _dtype(t):
    return {torch.float16: 0, torch.bfloat16: 1}[t.dtype]


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def attention_workspace_bytes(seqs, max_q, max_kv, hq, hkv, d, prompts=False):
    """Bytes that the attention wants in order to run contexts in pieces; 0: these sizes never do."""
    f = _entry("fq_attention_workspace_bytes", ctypes.c_size_t)
    return int(f(*_args(seqs, max_q, (max_kv,), hq, hkv, d, int(prompts))))


def attention_in_one_piece(q, kp, kn, vp, vn, c, r, is_causal=False):
    """fq_fused_tq_attention: the entry without a workspace, which never runs a context in pieces."""
    b, hq, nq, d = q.shape
    out, r = torch.empty_like(q), r.contiguous()
    st = _entry("fq_fused_tq_attention")(*_args(q, kp, kn, vp, vn, c, c, r, 0, out, b, hq, kp.shape[1], nq, kp.shape[2], d,
                                                d ** -0.5, int(is_causal), _dtype(q)), _stream())
    assert st == 0, st
    return out


def _pieces_room(seqs, max_q, max_kv, hq, hkv, d, prompts, dev):
    """A workspace that suffices for contexts in pieces and for nothing else, and its bytes."""
    n = int(_entry("fq_attention_pieces_workspace_bytes", ctypes.c_size_t)(*_args(seqs, max_q, (max_kv,), hq, hkv, d, prompts)))
    return torch.empty(n, dtype=torch.uint8, device=dev) if n else None, ctypes.c_size_t(n)


def attention_on_packed_rows(q, kp, kn, vp, vn, c, r, is_causal=False):
    """fq_fused_tq_attention_split with room for contexts in pieces alone: keys and values are not expanded first."""
    b, hq, nq, d = q.shape
    hkv, nkv = kp.shape[1:3]
    out, r = torch.empty_like(q), r.contiguous()
    ws, n = _pieces_room(b, nq, nkv, hq, hkv, d, 1 if is_causal else 2, q.device)
    st = _entry("fq_fused_tq_attention_split")(*_args(q, kp, kn, vp, vn, c, c, r, 0, out, b, hq, hkv, nq, nkv, (nkv,), (nkv,), d, d ** -0.5,
                                                      int(is_causal), _dtype(q), ws), n, _stream())
    assert st == 0, st
    return out


def prefill_on_packed_rows(q, cu, max_q, cache, table, sl, c, r, hkv, d, bs, causal=True, out=None):
    """fq_paged_tq4_prefill_split with room for contexts in pieces alone."""
    out, r = torch.zeros_like(q) if out is None else out, r.contiguous()
    ws, n = _pieces_room(table.shape[0], max_q, table.shape[1] * bs, q.shape[1], hkv, d, 0, q.device)
    st = _entry("fq_paged_tq4_prefill_split")(*_args(q, cu, cache, table, sl, c, c, r, 0, out, table.shape[0], max_q, q.shape[1], hkv, d, bs,
                                                     table.shape[1], (cache.shape[0],), d ** -0.5, int(causal), _dtype(q), (q.shape[0],), ws), n,
                                              _stream())
    assert st == 0, st
    return out


def prefill_in_one_piece(q, cu, max_q, cache, table, sl, c, r, hkv, d, bs, causal=True):
    """fq_paged_tq4_prefill: the paged entry without a workspace."""
    out, r = torch.zeros_like(q), r.contiguous()
    st = _entry("fq_paged_tq4_prefill")(*_args(q, cu, cache, table, sl, c, c, r, 0, out, table.shape[0], max_q, q.shape[1], hkv,
                                               d, bs, table.shape[1], (cache.shape[0],), d ** -0.5, int(causal), _dtype(q)), _stream())
    assert st == 0, st
    return out
