"""Float products with the gate's activation or the rotation and the cache write in the product's own kernel: the bits of the two kernels."""

import pytest
import torch

from tests.test_kernels_gpu import rnd

pytestmark = pytest.mark.gpu


def ops():
    from paged_llm_amd.csrc import ops as o
    return o


def each_tile(monkeypatch):
    """Every form of the kernel, whatever the sizes would choose."""
    for tile in ops().FLOAT_GEMM_TILES:
        monkeypatch.setattr(ops(), "float_gemm_plan", lambda *a, tile=tile: tile)
        yield tile


@pytest.mark.parametrize("m,ff,k", [(1, 8, 32), (9, 12, 100), (17, 129, 512), (50, 40, 2048)])
@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
def test_gated_float_product(m, ff, k, activation, monkeypatch):
    """Gate rows whose number is no multiple of eight, rows and weight rows past the last tile, a K with a tail."""
    o = ops()
    a, w = rnd(m, k, seed=1).cuda(), rnd(2 * ff, k, seed=2).cuda()
    want = o.gate_mul(o.gemm_generic(a, w), activation)
    for tile in each_tile(monkeypatch):
        assert torch.equal(o.gemm_float_gated(a, w, activation), want), tile


@pytest.mark.parametrize("heads,kv_heads,d,bs", [(4, 2, 64, 16), (3, 1, 48, 32), (2, 2, 16, 4)])
@pytest.mark.parametrize("m,k,turns", [(1, 64, True), (20, 512, True), (70, 96, False)])
def test_rotary_float_product(heads, kv_heads, d, bs, m, k, turns, monkeypatch):
    """Queries, keys and values against the product and the rotary kernel apart; a slot of -1 writes nothing."""
    o = ops()
    a, w = rnd(m, k, seed=3).cuda(), rnd((heads + 2 * kv_heads) * d, k, seed=4).cuda()
    g = torch.Generator().manual_seed(5)
    positions = torch.randint(0, 200, (m,), generator=g, dtype=torch.int32).cuda()
    slots = torch.randperm(4 * m, generator=g)[:m].to(torch.int32)
    slots[m // 2] = -1
    slots = slots.cuda()
    cos, sin = (rnd(200, d // 2, seed=s).cuda() for s in (6, 7)) if turns else (None, None)
    pages = 4 * m // bs + 1

    def cache():
        return torch.full((pages, kv_heads, bs, d), 7.0, device="cuda"), torch.full((pages, kv_heads, d, bs), 7.0, device="cuda")
    k1, v1 = cache()
    qkv = o.gemm_generic(a, w)
    o.rope_scatter(qkv, positions, cos, sin, heads, kv_heads, d, slots, k1, v1, bs, d if turns else 0)
    for tile in each_tile(monkeypatch):
        k2, v2 = cache()
        q = o.gemm_float_rotary(a, w, dict(positions=positions, cos=cos, sin=sin, slots=slots, k_pages=k2, v_pages=v2, num_heads=heads,
                                           num_kv_heads=kv_heads, head_dim=d, block_size=bs))
        assert torch.equal(q, qkv[:, :heads * d]) and torch.equal(k1, k2) and torch.equal(v1, v2), tile


@pytest.mark.parametrize("m,n,k", [(5, 20, 64), (40, 70, 2048), (33, 40, 50)])
def test_float_product_of_infinities_and_huge_numbers(m, n, k):
    """Infinities, NaN and numbers past the largest bfloat16 give what float arithmetic gives, and leave the other results alone; so do
    numbers so small that their parts lose bits, to an error below the smallest normal number's share."""
    o = ops()
    a, w = rnd(m, k, seed=8), rnd(n, k, seed=9)
    plain = o.gemm_generic(a.cuda(), w.cuda()).cpu()
    a[1, 3], w[2, k - 1], w[3, 0] = float("inf"), float("-inf"), float("nan")
    a[2, :], w[4, :] = 0.0, 0.0
    a[2, 5], w[4, 5] = 3.4e38, 0.5                               # rounds past the largest bfloat16; the result is finite
    a[3] *= 2.0 ** -120
    want = (a.double() @ w.double().T).float()
    for tile in o.FLOAT_GEMM_TILES:
        out = torch.empty(m, n, device="cuda")
        ga, gw = a.cuda(), w.cuda()
        assert o._fn("gemm_float.hip", "pllm_gemm_float")(ga.data_ptr(), k, 0, gw.data_ptr(), k, 0, out.data_ptr(), n, 0, m, n, k, 1, *tile, o._stream()) == 0
        out = out.cpu()
        odd = ~torch.isfinite(want)
        assert torch.equal(torch.isnan(out), torch.isnan(want)) and torch.equal(out[odd & ~torch.isnan(want)], want[odd & ~torch.isnan(want)])
        assert float(out[2, 4]) == float(want[2, 4])
        same = torch.ones(m, n, dtype=torch.bool)
        same[[1, 2, 3]], same[:, [2, 3, 4]] = False, False
        assert torch.equal(out[same], plain[same])
        ok = ~odd[3]
        assert float((out[3].double() - want[3].double())[ok].abs().max()) <= 2.0 ** -22 * float(want[3][ok].abs().max()) + k * 2.0 ** -133
