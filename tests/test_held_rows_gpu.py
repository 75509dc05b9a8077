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


def shifted(x):
    """The same numbers one element further on in memory: rows that no 16-byte boundary fits."""
    return torch.cat([x.new_zeros(1), x.reshape(-1)])[1:].view(x.shape)


@pytest.mark.parametrize("width", [1024, 1028, 2048, 4096])
@pytest.mark.parametrize("kind", ["rows", "choices", "pair", "none"])
def test_a_rows_bits_do_not_hang_on_where_it_lies(width, kind):
    """Four elements a load or one: the same partial sums in the same order, whatever stands in front of the norm."""
    from paged_llm_amd.csrc import ops
    rows, top = 3, 2
    stream, a, b = (rnd(rows, width, seed=s).cuda() for s in (1, 2, 3))
    wb, wn, bias = (rnd(width, seed=s).cuda() for s in (4, 5, 6))
    e, h, weights = rnd(rows * top, width, seed=7).cuda(), rnd(rows, width, seed=8).cuda(), rnd(rows, top, seed=9).cuda()
    places = torch.tensor([3, -1, 0, 5, 2, 1], dtype=torch.int32, device="cuda")

    def norm(place):
        s = place(stream.clone())
        branch = {"rows": lambda: place(a), "pair": lambda: ops.WeightedPair(place(a), 0.3, place(b), 1.7), "none": lambda: None,
                  "choices": lambda: ops.ChoiceSum(place(e), place(h), places, weights)}[kind]()
        out = place(torch.zeros_like(stream))
        ops.rms_sandwich(s, branch, None if kind == "none" else place(wb), 0.5, 1e-5, w_next=place(wn), out=out, bias=None if kind == "none" else place(bias))
        return s, out
    for x, y in zip(norm(lambda t: t), norm(shifted)):
        assert torch.equal(x, y)


@pytest.mark.parametrize("width", [1024, 4096])
def test_the_depth_norms_bits_do_not_hang_on_where_its_rows_go(width):
    """The tokens' own rows and the output may lie anywhere: which elements a thread sums follows from the float rows alone."""
    from paged_llm_amd.csrc import ops
    rows, top = 3, 2
    stream, h, wb, wn = rnd(rows, width, seed=1).cuda(), rnd(rows, width, seed=2).to(torch.bfloat16).cuda(), rnd(width, seed=3).cuda(), rnd(width, seed=4).cuda()
    e, weights = rnd(rows * top, width, seed=5).cuda(), rnd(rows, top, seed=6).cuda()
    places = torch.tensor([3, -1, 0, 5, 2, 1], dtype=torch.int32, device="cuda")

    def norm(own, out):
        s, history = stream.clone(), rnd(3, rows, width, seed=7).cuda()
        ops.rms_sandwich(s, ops.ChoiceSum(e, own, places, weights), wb, 0.5, 1e-5, w_next=wn, out=out, depth=ops.DepthSum(history, rnd(3, seed=8).cuda()))
        return s, history, out
    plain = norm(h, torch.zeros(rows, width, device="cuda", dtype=torch.bfloat16))
    for x, y in zip(plain, norm(shifted(h), torch.zeros(rows, width + 3, device="cuda", dtype=torch.bfloat16)[:, :width])):
        assert torch.equal(x, y)
