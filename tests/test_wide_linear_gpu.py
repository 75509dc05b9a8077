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


def test_silu_to_float_accuracy():
    """SiLU of gates that are exactly known floats (sums of three bfloat16 numbers, one product each) times one, rounded to bfloat16: a float's error of
    1.8e-7 crosses a rounding boundary in at most 1.8e-7 * 2^8 of the results.  Values past the fast form's range are those of the exponential function."""
    o = ops()
    n, m, k = 16, 20000, 64
    g = torch.Generator().manual_seed(11)
    z = (-80.0 + 50.0 * torch.rand(m, n, generator=g, dtype=torch.float64)).float()
    x, rest = torch.zeros(m, k, dtype=torch.bfloat16), z
    w = torch.zeros(2 * n, k, dtype=torch.bfloat16)
    for part in range(3):
        x[:, part * n:(part + 1) * n] = rest.to(torch.bfloat16)
        rest = rest - rest.to(torch.bfloat16).float()
        w[torch.arange(n), part * n + torch.arange(n)] = 1.0
    x[:, k - 1], w[n:, k - 1] = 1.0, 1.0
    special = torch.zeros(8, k, dtype=torch.bfloat16)            # a gate of its own in every row, one weight row that takes it
    special[:, 0] = torch.tensor([-3e38, float("-inf"), float("nan"), -87.5, -88.5, -95.0, -200.0, 100.0])
    special[:, k - 1] = 1.0
    w8 = torch.zeros(8, k, dtype=torch.bfloat16)
    w8[0, 0] = w8[4:, k - 1] = 1.0
    want = (z.double() / (1 + torch.exp(-z.double()))).to(torch.bfloat16)
    tiled, tiled8 = o.tile_weight(w.cuda(), "gated"), o.tile_weight(w8.cuda(), "gated")
    for tile in o.WIDE_TILES[:1] + o.WIDE_GATED_TILES[-1:]:
        got = o.wide_linear(x.cuda(), tiled, tile, o.SL_GATED).cpu()
        assert int((got != want).sum()) <= 1.8e-7 * 256 * m * n + 16, tile
        edge = o.wide_linear(special.cuda(), tiled8, tile, o.SL_GATED).cpu()[:, 0].float()
        zs = special[:, 0].float()
        exact = zs / (1 + torch.exp(-zs))
        assert torch.equal(torch.isnan(edge), torch.isnan(exact))
        ok = ~torch.isnan(exact)
        assert torch.equal(edge[ok].to(torch.bfloat16), exact[ok].to(torch.bfloat16)), (edge, exact)


@pytest.mark.parametrize("m,n,k", [(257, 188, 64), (321, 364, 128), (130, 16, 320), (300, 520, 1088)])
@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
def test_gated_products_in_large_tiles(m, n, k, activation):
    """Every large tile where its last rows, blocks, stages and pieces of 16 bytes are whole or not: the bits of the smallest tile (the same chains of sums), also
    of gates past the quick form's range and of rows that are no numbers, and nothing past the last row."""
    o = ops()
    x, w = bf(m, k, seed=31), bf(2 * n, k, seed=32) * 0.25
    x[3] *= 64.0
    x[m - 2, 0], x[m // 2, 1] = float("nan"), float("inf")
    tiled, gx = o.tile_weight(w.cuda(), "gated"), x.cuda()
    want = o.wide_linear(gx, tiled, (64, 64), o.SL_GATED, activation=activation).cpu()
    for tile in o.WIDE_LARGE_TILES:
        got = o.wide_linear(gx, tiled, tile, o.SL_GATED, activation=activation).cpu()
        assert torch.equal(got.nan_to_num(7.0, 8.0, 9.0), want.nan_to_num(7.0, 8.0, 9.0)), tile


@pytest.mark.parametrize("m,n,k", [(257, 292, 64), (321, 364, 128), (130, 16, 320), (300, 520, 1088)])
def test_plain_products_in_large_tiles(m, n, k):
    """As ``test_plain_products``, and the bits of the smallest tile."""
    o = ops()
    x, w = bf(m, k, seed=34), bf(n, k, seed=35)
    gx, tiled = x.cuda(), o.tile_weight(w.cuda())
    want = o.wide_linear(gx, tiled, (64, 64), o.SL_F32)
    for tile in o.WIDE_PLAIN_TILES:
        assert torch.equal(o.wide_linear(gx, tiled, tile, o.SL_F32), want), tile
        assert torch.equal(o.wide_linear(gx, tiled, tile, o.SL_BF16), want.to(torch.bfloat16)), tile


def test_rows_of_a_very_wide_matrix():
    """A tile's offsets have 32 bits: rows further apart than they reach are laid side by side first."""
    o = ops()
    x, w = bf(320, 64, seed=36), bf(512, 64, seed=37)
    wide = torch.empty((320, o.WIDE_LARGE_OFFSETS * 2), dtype=torch.bfloat16, device="cuda")
    wide[:, :64] = x.cuda()
    tiled = o.tile_weight(w.cuda())
    for tile in ((64, 64),) + o.WIDE_PLAIN_TILES:
        assert torch.equal(o.wide_linear(wide[:, :64], tiled, tile), o.wide_linear(x.cuda(), tiled, tile)), tile


@pytest.mark.parametrize("m,n,k,tile", [(1000, 5632, 1024, (256, 128)), (321, 512, 1024, (64, 64)), (290, 11264, 1024, (192, 128)), (2100, 5632, 1024, (192, 256)), (129, 2048, 1088, (64, 64))])
def test_parts_take_the_wide_kernel_for_gated_products_of_long_k(m, n, k, tile, monkeypatch):
    """n weight rows; within two roundings to bfloat16 of 64 bits."""
    from paged_llm_amd.parts.linear import Weight, gated_linear
    w = bf(n, k, seed=33) * 0.1
    weight = Weight(w.cuda(), "gated")
    for x, rows in rows_of_three_kinds(m, k):
        tiles = taken(monkeypatch)
        got = gated_linear(x, weight).cpu().double()
        assert tiles == [tile]
        sums = rows.double() @ w.cuda().double().T
        want = (torch.nn.functional.silu(sums[:, :n // 2]) * sums[:, n // 2:]).cpu()
        assert bool(((got - want).abs() <= 2.0 ** -7 * want.abs() + 1e-3 * want.abs().max()).all())
        monkeypatch.undo()


def taken(monkeypatch):
    """The tiles that the products of the parts go to in the wide kernel, from here on."""
    from paged_llm_amd.parts import linear as part
    tiles, real = [], part.ops.wide_linear
    monkeypatch.setattr(part.ops, "wide_linear", lambda x, w, tile, *a, **k: (tiles.append(tile), real(x, w, tile, *a, **k))[1])
    return tiles


def rows_of_three_kinds(m, k):
    """Rows as a part gets them: a matrix, rows that no 16-byte load can take, and a sum and norm still to be done; with what they are."""
    from paged_llm_amd.parts.norm import PendingNorm
    x, delta, weight = bf(m, k, seed=21).cuda(), bf(m, k, seed=22).cuda(), (1.0 + 0.1 * rnd(k, seed=23)).cuda()
    odd = torch.zeros(m, k + 1, dtype=torch.bfloat16, device="cuda")[:, 1:]
    odd.copy_(x)
    pending = PendingNorm(weight, 1e-5, x.clone(), delta)
    return [(x, x), (odd, x), (pending, ops().rmsnorm(x.clone(), weight, 1e-5, delta))]


@pytest.mark.parametrize("m,n,k,tile", [(200, 2048, 128, (64, 64)), (600, 2048, 64, (64, 128)), (128, 2048, 128, None), (600, 2048, 96, None), (600, 2044, 8256, None)])
def test_parts_take_the_wide_kernel_for_products(m, n, k, tile, monkeypatch):
    """From 129 rows on where its plan has a tile; float results within the roundings of k products, bfloat16 ones those rounded once."""
    from paged_llm_amd.parts.linear import Weight, linear
    w = bf(n, k, seed=24) * 0.25
    weight = Weight(w.cuda())
    for x, rows in rows_of_three_kinds(m, k):
        tiles = taken(monkeypatch)
        got = linear(x, weight, torch.float32).cpu()
        rows = rows.cpu().double()
        assert tiles == ([tile] if tile else [])
        assert bool(((got.double() - rows @ w.double().T).abs() <= (k + 32) * 2.0 ** -24 * (rows.abs() @ w.double().abs().T)).all())
        short = linear(x, weight).cpu()
        assert len(tiles) == (2 if tile else 0) and (not tile or torch.equal(short, got.to(torch.bfloat16)))
        monkeypatch.undo()


@pytest.mark.parametrize("m,n,tile", [(250, 2048, (64, 64)), (250, 8192, (128, 128)), (400, 5632, (192, 192)), (320, 5632, (128, 160)), (300, 8192, None), (2048, 5632, None)])
def test_parts_take_the_wide_kernel_for_gated_products(m, n, tile, monkeypatch):
    """Large tiles from 321 rows on (below, the tiled kernel has them), no second round; within two roundings to bfloat16 of 64 bits."""
    from paged_llm_amd.parts.linear import Weight, gated_linear
    k = 128
    w = bf(2 * n, k, seed=25) * 0.25
    weight = Weight(w.cuda(), "gated")
    for x, rows in rows_of_three_kinds(m, k):
        tiles = taken(monkeypatch)
        got = gated_linear(x, weight).cpu().double()
        assert tiles == ([tile] if tile else [])
        sums = rows.double() @ w.cuda().double().T
        want = (torch.nn.functional.silu(sums[:, :n]) * sums[:, n:]).cpu()
        assert bool(((got - want).abs() <= 2.0 ** -7 * want.abs() + 1e-3 * want.abs().max()).all())
        monkeypatch.undo()


@pytest.mark.parametrize("m,heads,kv_heads,tile", [(768, 32, 8, (96, 96)), (768, 32, 4, None), (264, 64, 16, (64, 128)), (256, 64, 16, None), (1600, 32, 4, (128, 160))])
def test_parts_take_the_wide_kernel_for_rotary_products(m, heads, kv_heads, tile, monkeypatch):
    """Where the tiled kernel has no tiles, and in full rounds of 96 x 96; queries, keys and values as the product and the rotary kernel apart give them."""
    from types import SimpleNamespace
    from paged_llm_amd.parts.linear import Weight, qkv_rotary_cache
    o = ops()
    d, k, bs = 64, 128, 16
    w = bf((heads + 2 * kv_heads) * d, k, seed=26).cuda()
    weight, turn = Weight(w, "rotary", d), SimpleNamespace(cos=rnd(m, d // 2, seed=6).cuda(), sin=rnd(m, d // 2, seed=7).cuda(), rotary_dim=0, interleaved=False)
    positions = torch.arange(m, dtype=torch.int32, device="cuda")

    def run(x, weight):
        kp, vp = torch.zeros(m // bs + 1, kv_heads, bs, d, dtype=torch.bfloat16, device="cuda"), torch.zeros(m // bs + 1, kv_heads, d, bs, dtype=torch.bfloat16, device="cuda")
        q = qkv_rotary_cache(x, weight, positions, turn, heads, kv_heads, d, positions, kp, vp, bs)
        return q[:, :heads * d].float(), kp.float(), vp.float()
    for x, rows in rows_of_three_kinds(m, k):
        want = run(rows, w)
        tiles = taken(monkeypatch)
        got = run(x, weight)
        assert tiles == ([tile] if tile else [])
        for a, b in zip(got, want):
            assert bool(((a - b).abs() <= 2.0 ** -6 * b.abs() + 2.0 ** -6 * b.abs().max() * 0.25).all())
        monkeypatch.undo()
