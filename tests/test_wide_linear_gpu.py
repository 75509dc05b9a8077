"""The wide kernel of prompt products: every tile and every epilogue at the edges of tiles, one to several stages."""

import pytest
import torch

from tests.test_kernels_gpu import rnd

pytestmark = pytest.mark.gpu


def ops():
    from paged_llm_amd.csrc import ops as o
    return o


def bf(*shape, seed):
    return rnd(*shape, seed=seed).to(torch.bfloat16)


SIZES = [(129, 100, 64), (257, 200, 128), (300, 16, 320), (193, 392, 1088)]


@pytest.mark.parametrize("m,n,k", SIZES)
def test_plain_products(m, n, k):
    """Float results within the roundings of a chain of k products (2^-24 of the sum of magnitudes each, plus one for every group of 32);
    bfloat16 results are those rounded once; nothing past the last row or column."""
    o = ops()
    x, w = bf(m, k, seed=1), bf(n, k, seed=2)
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    wide = torch.zeros(m, k + 8, dtype=torch.bfloat16)
    wide[:, :k] = x
    gx, tiled = wide.cuda()[:, :k], o.tile_weight(w.cuda())
    for tile in o.WIDE_TILES:
        got = o.wide_linear(gx, tiled, tile, o.SL_F32).cpu()
        assert bool(((got.double() - want).abs() <= (k + 32) * 2.0 ** -24 * size).all()), tile
        assert torch.equal(o.wide_linear(gx, tiled, tile, o.SL_BF16).cpu(), got.to(torch.bfloat16)), tile


@pytest.mark.parametrize("m,n,k", SIZES)
@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
def test_gated_products(m, n, k, activation):
    """n outputs (not all multiples of eight): within two roundings to bfloat16 of the gate of the float sums."""
    o = ops()
    x, w = bf(m, k, seed=3), bf(2 * n, k, seed=4) * 0.25
    sums = x.double() @ w.double().T
    want = torch.nn.functional.silu(sums[:, :n]) if activation == "silu" else torch.nn.functional.gelu(sums[:, :n], approximate="tanh")
    want = want * sums[:, n:]
    tiled = o.tile_weight(w.cuda(), "gated")
    for tile in o.WIDE_TILES + o.WIDE_GATED_TILES:
        got = o.wide_linear(x.cuda(), tiled, tile, o.SL_GATED, activation=activation).cpu().double()
        assert bool(((got - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4 * want.abs().max()).all()), tile


@pytest.mark.parametrize("heads,kv_heads,d,bs", [(4, 2, 64, 16), (3, 1, 48, 32), (2, 2, 16, 4)])
@pytest.mark.parametrize("m,k,turns", [(130, 64, True), (200, 320, False)])
def test_rotary_products(heads, kv_heads, d, bs, m, k, turns):
    """The bits of the tiled kernel's epilogue (the same chains of sums); a slot of -1 writes nothing."""
    o = ops()
    x, w = bf(m, k, seed=7).cuda(), bf((heads + 2 * kv_heads) * d, k, seed=8).cuda()
    g = torch.Generator().manual_seed(9)
    positions = torch.randint(0, 200, (m,), generator=g, dtype=torch.int32).cuda()
    slots = torch.arange(8, m + 8, dtype=torch.int32)
    slots[m // 2:] = (torch.randperm(2 * m, generator=g)[:m - m // 2] + 2 * m).to(torch.int32)
    slots[5] = -1
    slots = slots.cuda()
    cos, sin = (rnd(200, d // 2, seed=s).cuda() for s in (6, 7)) if turns else (None, None)
    tiled, pages = o.tile_weight(w, "rotary", d), 5 * m // bs + 1

    def run(product):
        kp, vp = torch.full((pages, kv_heads, bs, d), 7.0, device="cuda", dtype=torch.bfloat16), torch.full((pages, kv_heads, d, bs), 7.0, device="cuda", dtype=torch.bfloat16)
        q = product(dict(positions=positions, cos=cos, sin=sin, slots=slots, k_pages=kp, v_pages=vp, num_heads=heads, num_kv_heads=kv_heads, head_dim=d, block_size=bs))
        return q, kp, vp
    want = run(lambda rope: o.tile_linear(x, tiled, o.SL_ROPE_KV, rope=rope))
    for tile in o.WIDE_TILES:
        got = run(lambda rope: o.wide_linear(x, tiled, tile, o.SL_ROPE_KV, rope=rope))
        assert all(torch.equal(a, b) for a, b in zip(want, got)), tile
