"""Float attention with one and with four workgroups for a tile of columns: the same bits, at the edges of blocks, chains and groups."""

import pytest
import torch

from tests.test_kernels_gpu import paged_case

pytestmark = pytest.mark.gpu


def ops():
    from paged_llm_amd.csrc import ops as o
    return o


def both(monkeypatch, *args, **kw):
    o, got = ops(), []
    for cut in (1, 4):
        monkeypatch.setattr(o, "float_attention_plan", lambda *a, cut=cut: cut)
        got.append(o.paged_attention_float(*args, **kw))
    return got


# heads of one to sixteen tiles of 16; blocks of 32 keys up to 64, of 16 beyond
@pytest.mark.parametrize("heads,kv_heads,d,bs", [(32, 4, 64, 16), (3, 1, 16, 48), (6, 2, 80, 16), (2, 2, 128, 32), (5, 1, 256, 16)])
@pytest.mark.parametrize("lens,num_q", [([1], [1]), ([16, 32, 33], [1, 2, 1]), ([256, 257, 512, 513], [1, 1, 3, 1]), ([1040, 7], [40, 7])])
def test_both_cuts_give_the_same_bits(heads, kv_heads, d, bs, lens, num_q, monkeypatch):
    o = ops()
    q, kp, vp, tables, cu, sl = paged_case(lens, num_q, heads, kv_heads, d, bs, torch.float32, seed=1)
    args = (q.cuda(), kp.cuda(), vp.cuda(), tables.cuda(), cu.cuda(), sl.cuda(), heads, kv_heads, d, d ** -0.5)
    sinks = torch.linspace(-2.0, 3.0, heads).cuda()
    for window, terms, weights in ((0, None, None), (200, o.ScoreTerms(sinks=sinks), None), (-256, o.ScoreTerms(cap=4.0, sinks=sinks), None),
                                   (130, None, o.KeyWeights(keep_first=20)), (0, None, o.KeyWeights(sigmoid=True, head_bias=sinks))):
        one, four = both(monkeypatch, *args, window, terms=terms, weights=weights)
        want = o.paged_attention_generic(*args, window, terms=terms, weights=weights)
        assert torch.equal(one, four), window
        assert float((one - want).abs().max() / want.abs().max()) <= 4e-5, window            # (two orders of float sums of up to 1,040 terms)


def test_values_that_are_no_numbers(monkeypatch):
    """Unseen slots full of NaN change nothing, and an infinite value reaches the columns that see it alone."""
    heads, kv_heads, d, bs, lens, num_q = 8, 2, 64, 16, [130, 45], [70, 1]
    q, kp, vp, tables, cu, sl = paged_case(lens, num_q, heads, kv_heads, d, bs, torch.float32, seed=2)
    args = lambda v: (q.cuda(), kp.cuda(), v.cuda(), tables.cuda(), cu.cuda(), sl.cuda(), heads, kv_heads, d, 0.125)
    want = both(monkeypatch, *args(vp))[0]
    odd = vp.clone()
    for s, n in enumerate(lens):
        last = int(tables[s, (n - 1) // bs])
        odd[last, :, :, (n - 1) % bs + 1:] = float("nan")
    assert all(torch.equal(got, want) for got in both(monkeypatch, *args(odd)))
    at = 100                                                     # a position that the first sequence's tokens see from 100 on
    odd[int(tables[0, at // bs]), 0, 3, at % bs] = float("inf")
    for got in both(monkeypatch, *args(odd)):
        sees = torch.arange(70).cuda() + 60 >= at
        column = got[:70].view(70, heads, d)
        assert bool((column[sees][:, :4, 3] == float("inf")).all()) and torch.equal(got[70:], want[70:])
        column[:, :4, 3] = want[:70].view(70, heads, d)[:, :4, 3]
        assert torch.equal(got, want)


def test_which_cut():
    o = ops()
    plan = lambda q, seqs, keys, heads=32, kv=4, d=64: o.float_attention_plan(q, seqs, heads, kv, d, 0, keys, 256)
    assert plan(8, 8, 700) == plan(1, 1, 180) == plan(61, 61, 2000) == plan(8, 8, 512, 16, 1, 256) == 4
    assert plan(12, 12, 100) == plan(301, 1, 301) == plan(64, 1, 64) == plan(128, 1, 128) == plan(2000, 1, 2000) == 1


def test_short_windows_are_one_workgroups():
    """The kernel has one form for windows that reach up to 128 positions, so no place is set aside for the parts of four workgroups."""
    o = ops()
    plan = lambda window, q=8, seqs=8, heads=32, kv=4, d=64: o.float_attention_plan(q, seqs, heads, kv, d, window, 2000, 256)
    for window in (1, 16, 100, 128):
        assert plan(window) == plan(-window) == plan(window, 1, 1, 16, 1, 256) == 1
    assert plan(0) == plan(1024) == 4


def test_portions_behind_a_context_take_the_form_that_was_ahead():
    o = ops()
    plan = lambda q, keys, heads=32, kv=4, d=64: o.float_attention_plan(q, 1, heads, kv, d, 0, keys, 256)
    assert plan(100, 600) == plan(301, 301) == plan(200, 1200, 16, 1, 256) == plan(200, 200, 16, 1, 256) == 1
    assert plan(25, 1025) == plan(50, 1050) == plan(33, 2033) == plan(100, 1100, 16, 1, 256) == plan(100, 1100, 16, 8, 128) == 4
