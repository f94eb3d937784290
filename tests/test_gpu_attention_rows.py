"""How the attention kernels rotate, store and split their query rows: edges of the 32-row blocks,
either layout of the rotation matrix, outputs that are not 16-byte aligned."""
from __future__ import annotations

import pytest
import torch

from flashquant_amd import kernels as K
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
