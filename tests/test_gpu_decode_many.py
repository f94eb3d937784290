"""Paged decode of more sequences than a wavefront has lanes: token chunks sized from the actual lengths, four sequences a lane."""
from __future__ import annotations

import random

import pytest
import torch

from flashquant_amd import kernels as K
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
    assert (got[sl == 0] == 0).all()
