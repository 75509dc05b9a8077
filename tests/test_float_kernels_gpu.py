"""The kernels of the true 32-bit path on the float matrix cores, at the edges of their tiles: products in every form of the
kernel, attention with every mask, term and weighting, and values that are no numbers where nobody may see them."""

import math

import pytest
import torch

from tests.test_kernels_gpu import dense_attention, paged_case, rnd

pytestmark = pytest.mark.gpu


def ops():
    from paged_llm_amd.csrc import ops as o
    return o


@pytest.mark.parametrize("m,n,k", [(1, 16, 32), (17, 33, 31), (49, 65, 50), (65, 129, 513), (16, 64, 2047), (48, 64, 2048), (7, 70, 5632)])
def test_float_product_in_every_form(m, n, k):
    """Every tile gives the same bits.  Bound: a result is reached by at most ceil(K / 512) * 32 products in one chain, one
    addition of a pair and seven of the pairs, each rounded once (2^-24), so its error is at most that many roundings of the
    sum of the products' magnitudes."""
    o = ops()
    a, w = rnd(m, k, seed=1), rnd(n, k, seed=2)
    want, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    chain = -(-k // 512) * 32 + 8
    outs = []
    for tile in o.FLOAT_GEMM_TILES:
        for shift in (0, 1):                                    # rows that 16-byte loads can read, and rows that they cannot
            base_a, base_w = torch.zeros(m, k + 4 + shift), torch.zeros(n, k + 8 + shift)
            base_a[:, shift:k + shift], base_w[:, shift:k + shift] = a, w
            ga, gw, out = base_a.cuda()[:, shift:k + shift], base_w.cuda()[:, shift:k + shift], torch.full((m + 1, n), 7.0, device="cuda")
            code = o._fn("gemm_float.hip", "pllm_gemm_float")(ga.data_ptr(), ga.stride(0), 0, gw.data_ptr(), gw.stride(0), 0, out.data_ptr(), n, 0,
                                                              m, n, k, 1, *tile, o._stream())
            assert code == 0 and bool((out[m] == 7.0).all()), tile
            outs.append(out[:m].cpu())
    assert all(torch.equal(outs[0], x) for x in outs)
    assert bool(((outs[0].double() - want).abs() <= chain * 2.0 ** -24 * size + 1e-30).all())


@pytest.mark.parametrize("m,n,k", [(300, 16, 32), (70, 130, 64), (33, 260, 96), (40, 9, 480), (129, 600, 7)])
def test_float_product_of_short_rows_in_every_form(m, n, k):
    """One, two, three and fifteen slices with columns, each with as many wavefronts; one tile of weight rows, groups of eight tiles that
    are not full, and the bound above."""
    test_float_product_in_every_form(m, n, k)


@pytest.mark.parametrize("t,heads,n,k", [(700, 9, 64, 64), (130, 3, 128, 40), (5, 16, 512, 128)])
def test_float_products_of_heads_at_several_tiles(t, heads, n, k):
    """Rows and weight rows of several tiles in every head's product.  Bound: as for one product."""
    o = ops()
    a, w = rnd(t, heads, k, seed=5), rnd(heads, n, k, seed=6)
    got = o.gemm_heads(a.cuda(), o.HeadMatrices(w.cuda())).cpu().double()
    for h in range(heads):
        want, size = a[:, h].double() @ w[h].double().T, a[:, h].double().abs() @ w[h].double().abs().T
        assert bool(((got[:, h] - want).abs() <= 40 * 2.0 ** -24 * size + 1e-30).all()), h


def test_float_product_batches():
    """Heads side by side in the rows, one matrix each, written into wider rows."""
    o = ops()
    a, w = rnd(21, 5, 96, seed=3), rnd(5, 40, 96, seed=4)
    out = torch.zeros(21, 5, 43, device="cuda")
    o.gemm_heads(a.cuda(), o.HeadMatrices(w.cuda()), out=out[:, :, :40])
    want = torch.einsum("thk,hnk->thn", a.double(), w.double())
    assert float((out[:, :, :40].cpu().double() - want).abs().max() / want.abs().max()) <= 1e-6 and bool((out[:, :, 40:] == 0).all())


CASES = [([1], [1]), ([40, 9, 64], [8, 1, 3]), ([129, 300, 17], [129, 300, 17]), ([1000, 33, 2048, 5], [1, 1, 1, 1]), ([577, 64, 77], [37, 2, 12])]
SHAPES = [(32, 4, 64, 16), (3, 1, 48, 32), (5, 5, 16, 16), (6, 2, 128, 16), (40, 1, 144, 16), (2, 1, 256, 64)]


@pytest.mark.parametrize("heads,kv_heads,d,bs", SHAPES)
@pytest.mark.parametrize("lens,num_q", CASES)
def test_float_attention(heads, kv_heads, d, bs, lens, num_q):
    """Against the plain kernel in float32 (both within 2e-5 of dense attention in the tests of that kernel)."""
    o = ops()
    if sum(lens) * heads * d > 3_000_000 and heads != 32:
        pytest.skip("long case kept for one shape")
    q, kp, vp, tables, cu, sl = paged_case(lens, num_q, heads, kv_heads, d, bs, torch.float32, seed=1)
    args = (q.cuda(), kp.cuda(), vp.cuda(), tables.cuda(), cu.cuda(), sl.cuda(), heads, kv_heads, d, 1 / math.sqrt(d))
    g = torch.Generator().manual_seed(5)
    slopes, sinks = (torch.randn(heads, generator=g).mul(0.05).cuda() for _ in range(2))
    for window, terms, weights in ((0, None, None), (19, None, None), (-64, o.ScoreTerms(sinks=sinks), None), (100, o.ScoreTerms(cap=3.0, slopes=slopes, sinks=sinks), None),
                                   (70, None, o.KeyWeights(keep_first=4)), (33, o.ScoreTerms(cap=5.0), o.KeyWeights(keep_first=20, sigmoid=True, head_bias=sinks)),
                                   (0, None, o.KeyWeights(sigmoid=True))):
        got = o.paged_attention_float(*args, window, terms=terms, weights=weights)
        want = o.paged_attention_generic(*args, window, terms=terms, weights=weights)
        assert float((got - want).abs().max() / want.abs().max()) <= 4e-5, (window, terms, weights)
    want = dense_attention(q, kp, vp, tables, cu, sl, heads, kv_heads, d, 1 / math.sqrt(d))
    got = o.paged_attention_float(*args).cpu()
    assert float((got - want).abs().max() / want.abs().max()) <= 2e-5


def test_float_attention_does_not_depend_on_the_cut():
    """The same positions as one prompt, in portions and beside other requests: the same bits."""
    o = ops()
    heads, kv_heads, d, bs = 8, 2, 64, 16
    q, kp, vp, tables, cu, sl = paged_case([530], [530], heads, kv_heads, d, bs, torch.float32, seed=2)
    rest = (kp.cuda(), vp.cuda())
    for window, weights in ((0, None), (100, None), (90, o.KeyWeights(keep_first=5)), (100, o.KeyWeights(sigmoid=True))):
        tail = (heads, kv_heads, d, 0.125, window)
        whole = o.paged_attention_float(q.cuda(), *rest, tables.cuda(), cu.cuda(), sl.cuda(), *tail, weights=weights).cpu()
        for lo, hi in ((0, 1), (3, 70), (64, 128), (529, 530), (200, 467)):
            two = torch.cat([q[lo:hi], q[hi - 1:hi]]).cuda()
            part = o.paged_attention_float(two, *rest, tables.repeat(2, 1).cuda(), torch.tensor([0, hi - lo, hi - lo + 1], dtype=torch.int32, device="cuda"),
                                           torch.tensor([hi, hi], dtype=torch.int32, device="cuda"), *tail, weights=weights).cpu()
            assert torch.equal(part[:hi - lo], whole[lo:hi]) and torch.equal(part[hi - lo:], whole[hi - 1:hi]), (window, lo, hi)


@pytest.mark.parametrize("window", [1, 32, 33, 64, 128, 129, -32, -64, -128, -129])
@pytest.mark.parametrize("heads,kv_heads,d", [(3, 3, 64), (8, 2, 128), (4, 4, 16)])
def test_float_attention_of_short_windows(heads, kv_heads, d, window):
    """Windows on both sides of the lengths from which a workgroup has more wavefronts: a portion and single tokens against the plain kernel
    (bound as above), and the same bits for a position however it was cut."""
    o = ops()
    bs, n = 16, 391
    q, kp, vp, tables, cu, sl = paged_case([n], [n], heads, kv_heads, d, bs, torch.float32, seed=6)
    rest, tail = (kp.cuda(), vp.cuda()), (heads, kv_heads, d, d ** -0.5, window)
    for weights in (None, o.KeyWeights(sigmoid=True)) + ((o.KeyWeights(keep_first=70),) if window > 0 else ()):
        args = (q.cuda(), *rest, tables.cuda(), cu.cuda(), sl.cuda(), *tail)
        whole, want = o.paged_attention_float(*args, weights=weights), o.paged_attention_generic(*args, weights=weights)
        assert float((whole - want).abs().max() / want.abs().max()) <= 4e-5
        for lo, hi in ((0, 1), (127, 130), (255, 256), (n - 1, n), (60, 200)):
            part = o.paged_attention_float(q[lo:hi].cuda(), *rest, tables.cuda(), torch.tensor([0, hi - lo], dtype=torch.int32, device="cuda"),
                                           torch.tensor([hi], dtype=torch.int32, device="cuda"), *tail, weights=weights)
            assert torch.equal(part, whole[lo:hi]), (lo, hi)


def test_float_attention_leaves_unseen_slots_alone():
    """Garbage past the context, in table entries past it and in front of a window changes nothing; an infinite value reaches
    the queries that see its key and no other."""
    o = ops()
    heads, kv_heads, d, bs = 4, 2, 32, 16
    q, kp, vp, tables, cu, sl = paged_case([37, 5], [20, 1], heads, kv_heads, d, bs, torch.float32, seed=3)
    def run(kp, vp, tables, window):
        return o.paged_attention_float(q.cuda(), kp.cuda(), vp.cuda(), tables.cuda(), cu.cuda(), sl.cuda(), heads, kv_heads, d, 0.3, window).cpu()
    t2, kp2, vp2 = tables.clone(), kp.clone(), vp.clone()
    t2[1, 1:] = 999_999
    kp2[tables[1, 0], :, 5:, :] = float("nan")
    vp2[tables[1, 0], :, :, 5:] = float("inf")
    kp2[tables[0, 2], :, 5:, :] = float("nan")
    vp2[tables[0, 2], :, :, 5:] = float("nan")
    assert torch.equal(run(kp, vp, tables, 0), run(kp2, vp2, t2, 0))
    vp2[tables[0, 0], :, :, :14] = float("nan")                 # (positions that a window of 4 has passed before the first query, at 17)
    assert torch.equal(run(kp, vp, tables, 4), run(kp2, vp2, t2, 4))
    vp3 = vp.clone()
    vp3[tables[0, 1], :, 7, 13] = float("inf")                  # position 29 of the first request, channel 7
    plain, odd = run(kp, vp, tables, 0), run(kp, vp3, tables, 0)
    seen = torch.zeros(21, heads, d, dtype=torch.bool)
    seen[29 - 17:20, :, 7] = True
    assert bool(torch.isinf(odd.view(21, heads, d)[seen]).all()) and torch.equal(odd.view(21, heads, d)[~seen], plain.view(21, heads, d)[~seen])
