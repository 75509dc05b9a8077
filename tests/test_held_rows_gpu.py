"""The norm kernel that holds a row in registers, at the edges of its forms: one to four groups of four elements a thread, single elements (a
width that is no multiple of four, rows that do not lie on 16-byte boundaries), branches that are sums of few and of many choices, picked rows."""

import pytest
import torch

from tests.test_kernels_gpu import rnd

pytestmark = pytest.mark.gpu


def unit(x, eps=1e-5):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


@pytest.mark.parametrize("width,pad", [(4, 0), (1024, 0), (1028, 0), (2048, 0), (2048, 3), (2052, 8), (4096, 0), (4095, 0), (1022, 2)])
@pytest.mark.parametrize("top", [1, 4, 5, 70])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_sums_of_choices(width, pad, top, dtype):
    """Against 64 bits: float sums of `width` squares and `top` products, so 1e-5 in float32, and in bfloat16 half a step on top: a number
    of 8 bits is rounded by at most half of its last one, 2^-8 of itself just above a power of two."""
    from paged_llm_amd.csrc import ops
    rows = 5
    stream, e, h = rnd(rows, width, seed=1).cuda(), rnd(rows * top, width, seed=2).cuda(), rnd(rows, width + pad, seed=3).to(dtype).cuda()[:, :width]
    g = torch.Generator().manual_seed(4)
    places = torch.randperm(rows * top, generator=g).to(torch.int32)
    places[torch.randperm(rows * top, generator=g)[:rows]] = -1              # (some tokens hand their own row back)
    weights, wb, wn = rnd(rows, top, seed=5), rnd(width, seed=6), rnd(width, seed=7)
    out = torch.zeros(rows, width + pad, dtype=dtype, device="cuda")[:, :width]
    ops.rms_sandwich(stream, ops.ChoiceSum(e, h, places.cuda(), weights.cuda()), wb.cuda(), 0.5, 1e-5, w_next=wn.cuda(), out=out)
    picked = torch.where(places.view(rows, top, 1) >= 0, e.cpu().double()[places.clamp(min=0).long()].view(rows, top, width), h.cpu().double()[:, None, :])
    want = rnd(rows, width, seed=1).double() + 0.5 * unit((weights.double()[..., None] * picked).sum(1)) * wb.double()
    assert torch.allclose(stream.cpu().double(), want, rtol=1e-5, atol=1e-5)
    near = unit(want) * wn.double()
    assert torch.allclose(out.cpu().double(), near, rtol=1e-5 + (2.0 ** -8 if dtype == torch.bfloat16 else 0.0), atol=2e-5)


@pytest.mark.parametrize("width", [4, 1028, 4096, 4098, 2047])
def test_picked_rows_without_a_branch(width):
    from paged_llm_amd.csrc import ops
    x, w = rnd(9, width, seed=1), rnd(width, seed=2)
    pick = torch.tensor([8, 0, 3, 3], dtype=torch.int32)
    s = x.cuda()
    for index, rows in ((None, x), (pick, x[pick.long()])):
        got = ops.rms_sandwich(s, None, None, 0.0, 1e-5, w_next=w.cuda(), out_dtype=torch.float32, row_index=None if index is None else index.cuda())
        assert torch.allclose(got.cpu().double(), unit(rows.double()) * w.double(), rtol=1e-5, atol=1e-5)
        assert torch.equal(ops.rms_sandwich(s, None, None, 0.0, 1e-5, out_dtype=torch.bfloat16, row_index=None if index is None else index.cuda()).cpu(),
                           rows.to(torch.bfloat16))
    assert torch.equal(s.cpu(), x)
