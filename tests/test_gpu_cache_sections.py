"""Operators that read or write the sections of paged token rows in place, against the same operators on
contiguous copies of those sections (bit for bit)."""
import math

import pytest
import torch

from flashquant_amd import kernels as K
from flashquant_amd.vllm.impl import TQ4AttentionKernels

pytestmark = pytest.mark.gpu
DEV = "cuda"


def random_cache(pages, page, h, d, seed):
    g = torch.Generator().manual_seed(seed)
    row = h * (d + 8)
    cache = torch.randint(0, 256, (pages, page, row), dtype=torch.uint8, generator=g)
    flat = cache.view(-1, row)
    n = flat.shape[0]
    sections = []
    for first in (0, h * (d // 2 + 4)):
        norms = torch.rand(n, h, generator=g) * 30 + 0.01
        flat[:, first + h * d // 2: first + h * (d // 2 + 4)] = norms.view(torch.uint8)
        sections += [flat[:, first: first + h * d // 2].reshape(n, h, d // 2).contiguous(), norms.view(n, h, 1)]
    return cache.to(DEV), [t.to(DEV) for t in sections]


# one token, a tile that ends inside a token, several tiles of a workgroup, heads that do not divide a tile, more heads than
# 16 bits count
@pytest.mark.parametrize("pages,page,h", [(1, 1, 1), (3, 16, 1), (1, 8, 3), (5, 16, 8), (200, 32, 8), (7, 16, 40), (40, 16, 5), (2, 3, 70001)])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_decompress_cache_equals_decompress_of_its_sections(pages, page, h, d):
    layer = TQ4AttentionKernels(h, d, 1.0 / math.sqrt(d), torch.device(DEV))
    cache, (kp, kn, vp, vn) = random_cache(pages, page, h, d, 7 * pages + h + d)
    for dtype in (torch.bfloat16, torch.float16):
        for rotate in (True, False):
            k, v = layer.decompress_cache(cache, dtype, apply_rotation=rotate)
            assert k.shape == v.shape == (pages, page, h, d) and k.dtype == dtype
            for got, p, n in ((k, kp, kn), (v, vp, vn)):
                want = (K.tq4_decompress_rotated(p, n, layer.centroids, layer.rotation, dtype) if rotate
                        else K.tq4_decompress(p, n, layer.centroids, dtype))
                assert torch.equal(got.view(-1, h, d), want)
    k, v = layer.decompress_cache(cache, torch.float32, apply_rotation=False)
    assert torch.equal(v.view(-1, h, d), K.tq4_decompress(vp, vn, layer.centroids, torch.float32))
    # given outputs are written in place, a little beyond them stays as it is
    n = pages * page * h * d
    big = torch.full((2, n + 64), 7.0, dtype=torch.bfloat16, device=DEV)
    k, v = layer.decompress_cache(cache, torch.bfloat16, out_k=big[0], out_v=big[1])
    assert k.data_ptr() == big.data_ptr() and (big[:, n:] == 7).all()
    assert torch.equal(v.view(-1, h, d), K.tq4_decompress_rotated(vp, vn, layer.centroids, layer.rotation, torch.bfloat16))


# rows of 256 coordinates: the fewest that run in the pipelined form (64 a CU), one more and one fewer, last tiles of 1, 63 and 64
# rows, one tile and several a workgroup
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tiles,extra", [(1, -1), (1, 0), (1, 1), (2, -1), (3, 0), (3, 63), (4, 65)])
def test_decompress_rotated_of_many_wide_rows(tiles, extra, dtype):
    """The same bits as the same rows a few thousand at a time, which the other tests hold against a float32 product."""
    layer = TQ4AttentionKernels(1, 256, 1.0 / 16, torch.device(DEV))
    n = 64 * tiles * torch.cuda.get_device_properties(0).multi_processor_count + extra
    g = torch.Generator(device=DEV).manual_seed(n)
    packed = torch.randint(0, 256, (n, 1, 128), dtype=torch.uint8, generator=g, device=DEV)
    norms = torch.rand(n, 1, 1, generator=g, device=DEV) * 30 + 0.01
    for rotation in (layer.rotation.contiguous(), layer.rotation.t().contiguous().t()):
        out = torch.full((n + 1, 1, 256), 7.0, dtype=dtype, device=DEV)
        K.tq4_decompress_rotated(packed, norms, layer.centroids, rotation, dtype, out=out[:n])
        want = torch.cat([K.tq4_decompress_rotated(packed[i:i + 4001], norms[i:i + 4001], layer.centroids, rotation, dtype)
                          for i in range(0, n, 4001)])
        assert torch.equal(out[:n], want) and (out[n] == 7).all()
    # a cache row of one head: keys and values side by side
    cache = torch.cat([packed.view(n, 128), norms.view(n, 1).view(torch.uint8).view(n, 4)] * 2, dim=1).view(n, 1, 264)
    k, v = layer.decompress_cache(cache, dtype)
    assert torch.equal(k.view_as(want), want) and torch.equal(v.view_as(want), want)


def test_decompress_cache_of_no_pages_and_argument_errors():
    layer = TQ4AttentionKernels(8, 128, 1.0, torch.device(DEV))
    k, v = layer.decompress_cache(torch.empty(0, 16, 8 * 136, dtype=torch.uint8, device=DEV), torch.bfloat16)
    assert k.shape == v.shape == (0, 16, 8, 128)
    with pytest.raises(ValueError):
        layer.decompress_cache(torch.zeros(1, 16, 8 * 136, dtype=torch.uint8, device=DEV), torch.float32)
    with pytest.raises(ValueError):
        layer.decompress_cache(torch.zeros(1, 16, 7 * 136, dtype=torch.uint8, device=DEV), torch.bfloat16)


@pytest.mark.parametrize("n,h", [(1, 8), (3, 1), (130, 8), (9, 24)])
@pytest.mark.parametrize("d", [64, 128])
def test_prod_store_rows_writes_the_rows_and_nothing_else(n, h, d):
    g = torch.Generator().manual_seed(n + h)
    pages, page = n // 16 + 2, 16
    kn, kg, vi, vn, row = K.prod_page_layout(h, d)
    cache = torch.randint(0, 256, (pages, page, row), dtype=torch.uint8, generator=g)
    slots = torch.randperm(pages * page, generator=g)[:n]
    slots[0] = slots[0] - pages * page                      # counted from the end, as an indexed store does
    packed = [torch.randint(0, 256, (n, h, d // 2), dtype=torch.uint8, generator=g) for _ in range(2)]
    norms = [torch.rand(n, h, 1, generator=g) for _ in range(3)]
    want = cache.clone().view(-1, row)
    want[slots, :kn] = packed[0].view(n, -1)
    for at, t in ((kn, norms[0]), (kg, norms[1]), (vn, norms[2])):
        want[slots, at: at + 4 * h] = t.view(n, h).view(torch.uint8)
    want[slots, vi:vn] = packed[1].view(n, -1)
    got = cache.to(DEV)
    dev = [t.to(DEV) for t in (slots, packed[0], norms[0], norms[1], packed[1], norms[2])]
    K.prod_store_rows(got, *dev)
    assert torch.equal(got.cpu().view(-1, row), want)


# rows further apart than their bytes, a cache that starts at an odd byte, rows whose sections are no whole words
@pytest.mark.parametrize("h,d,gap,start", [(8, 128, 32, 0), (8, 128, 3, 0), (8, 128, 0, 1), (1, 66, 0, 0), (3, 10, 5, 2)])
def test_prod_store_rows_of_any_alignment_and_row_stride(h, d, gap, start):
    g = torch.Generator().manual_seed(h + d + gap)
    n, pages, page = 37, 4, 16
    kn, kg, vi, vn, row = K.prod_page_layout(h, d)
    buf = torch.randint(0, 256, (start + pages * page * (row + gap),), dtype=torch.uint8, generator=g)
    slots = torch.randperm(pages * page, generator=g)[:n]
    packed = [torch.randint(0, 256, (n, h, d // 2), dtype=torch.uint8, generator=g) for _ in range(2)]
    norms = [torch.rand(n, h, 1, generator=g) for _ in range(3)]

    def cache_of(b):
        return b[start:].view(pages, page, row + gap)[:, :, :row]

    want = buf.clone()
    flat = cache_of(want).view(-1, row)
    flat[slots] = torch.cat([packed[0].view(n, -1), norms[0].view(n, h).view(torch.uint8), norms[1].view(n, h).view(torch.uint8),
                             packed[1].view(n, -1), norms[2].view(n, h).view(torch.uint8)], dim=1)
    got = buf.to(DEV)
    dev = [t.to(DEV) for t in (slots, packed[0], norms[0], norms[1], packed[1], norms[2])]
    K.prod_store_rows(cache_of(got), *dev)
    assert torch.equal(got.cpu(), want)


def test_decompress_cache_at_an_odd_byte():
    layer = TQ4AttentionKernels(2, 64, 1.0, torch.device(DEV))
    cache, _ = random_cache(3, 16, 2, 64, 5)
    moved = torch.zeros(cache.numel() + 1, dtype=torch.uint8, device=DEV)[1:].view_as(cache)
    moved.copy_(cache)
    for rotate in (True, False):
        for a, b in zip(layer.decompress_cache(moved, torch.bfloat16, apply_rotation=rotate),
                        layer.decompress_cache(cache, torch.bfloat16, apply_rotation=rotate)):
            assert torch.equal(a, b)


def _prod_rows(n, h, d, seed):
    g = torch.Generator().manual_seed(seed)
    packed = [torch.randint(0, 256, (n, h, d // 2), dtype=torch.uint8, generator=g) for _ in range(2)]
    norms = [torch.rand(n, h, 1, generator=g) for _ in range(3)]
    row = torch.cat([packed[0].view(n, -1), norms[0].view(n, h).view(torch.uint8), norms[1].view(n, h).view(torch.uint8),
                     packed[1].view(n, -1), norms[2].view(n, h).view(torch.uint8)], dim=1)
    return (packed[0], norms[0], norms[1], packed[1], norms[2]), row


@pytest.mark.parametrize("form", ["one row", "slots in rows", "int packed", "strided bytes", "two-dimensional slots"])
def test_prod_store_rows_of_unusual_forms(form):
    """What an indexed store of assembled rows takes: one row for several slots, slots of more dimensions, indices of another
    integer type, a cache whose bytes lie apart."""
    h, d, pages, page = 4, 64, 3, 16
    n = 1 if form == "one row" else 6
    operands, row = _prod_rows(n, h, d, 7)
    slots = torch.tensor([3, 41, 17, -1, 8, 30])
    if form in ("slots in rows", "two-dimensional slots"):
        slots = slots[None] if form == "slots in rows" else torch.stack([slots, (slots + 1) % 48])
    gap = 2 if form == "strided bytes" else 1
    buf = torch.randint(0, 256, (pages, page, row.shape[1] * gap), dtype=torch.uint8, generator=torch.Generator().manual_seed(8))
    want = buf.clone()
    want[..., ::gap].view(-1, row.shape[1])[slots] = row
    got = buf.to(DEV)
    dev = [t.to(DEV) for t in operands]
    if form == "int packed":
        dev[0], dev[3] = dev[0].int(), dev[3].long()
    K.prod_store_rows(got[..., ::gap], slots.to(DEV), *dev)
    assert torch.equal(got.cpu(), want)


def test_prod_store_rows_skips_slots_outside_the_cache():
    h, d, pages, page = 2, 64, 2, 16
    operands, row = _prod_rows(5, h, d, 9)
    slots = torch.tensor([32, 4, -33, 1 << 40, 31])
    cache = torch.randint(0, 256, (pages, page, row.shape[1]), dtype=torch.uint8, generator=torch.Generator().manual_seed(10))
    want = cache.clone()
    want.view(-1, row.shape[1])[slots[[1, 4]]] = row[[1, 4]]
    got = cache.to(DEV)
    K.prod_store_rows(got, slots.to(DEV), *[t.to(DEV) for t in operands])
    assert torch.equal(got.cpu(), want)
