"""The experts' products for inner sizes that are multiples of 64 (tiles of 128 rows x 128 or 256 weight rows, of 64 rows x 128 or of
16 rows x 64, both operands through LDS in stages): against float64 sums of the same bfloat16 operands, and the same bits whatever the tile."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# inner size: one stage, fewer and more than the stages under way; outputs: no multiple of 16 or of a tile, one and several groups of 8
# tiles; tokens: experts with tiles of 1 to 128 rows; (777 and 1,178 tokens take tiles of 256 weight rows for gated and down products;
# 131 tokens of one expert take, with tiles of 16 rows, the kernel that cuts K between wavefronts, which adds in another order; the
# last case's weights are let go by the caches)
@pytest.mark.parametrize("tokens,top,experts,inner,outputs", [(300, 2, 8, 128, 192), (517, 2, 3, 192, 328), (260, 4, 5, 64, 72), (131, 1, 1, 448, 40),
                                                              (64, 3, 3, 320, 1100), (777, 2, 8, 192, 2040), (1178, 2, 8, 64, 2048),
                                                              (40, 2, 8, 1024, 1400)])
def test_staged_products(tokens, top, experts, inner, outputs):
    from paged_llm_amd.csrc import ops
    gen = torch.Generator().manual_seed(tokens)
    h = torch.randn((tokens, inner), generator=gen).to(torch.bfloat16).cuda()
    w = (torch.randn((experts, 2 * outputs, inner), generator=gen) * inner ** -0.5).to(torch.bfloat16).cuda()
    ids = torch.stack([torch.randperm(experts + 1, generator=gen)[:top] for _ in range(tokens)]).to(torch.int32).cuda()    # (expert `experts`: passed through)
    scale = torch.rand((tokens * top,), generator=gen).cuda()
    count = int((ids < experts).sum())
    for form in ("gated", "plain", "down"):
        got, want, spread = {}, None, None
        for rows in (ops.MOE_TILE_ROWS, ops.MOE_MID_TILE_ROWS, ops.MOE_MAX_TILE_ROWS):
            sorted_pair, row_of_pair, tiles = ops.moe_align(ids, experts, rows)
            place = row_of_pair.long()
            if form == "down":          # the rows of the pairs, each at the place this alignment gives it
                x = torch.zeros((tokens * top, inner), dtype=torch.bfloat16, device="cuda")
                x[place[place >= 0]] = h[torch.nonzero(place >= 0)[:, 0] // top] * scale[place >= 0, None].to(torch.bfloat16)
                out = ops.moe_expert_gemm(x, w, tiles, sorted_pair, top, False, tile_rows=rows)
            else:
                weights = w if form == "gated" else w[:, :outputs].contiguous()
                out = ops.moe_expert_gemm(h, weights, tiles, sorted_pair, top, form == "gated", "silu" if form == "gated" else "relu2", tile_rows=rows,
                                          pair_scale=scale if form == "gated" else None, plain=form == "plain")
            got[rows] = out[place[place >= 0]]
            if want is None:            # pair by pair in float64, with the sums of magnitudes that bound a float sum's error
                pair = torch.nonzero(place >= 0)[:, 0]
                rows_of_pairs = (x[place[pair]] if form == "down" else h[pair // top]).double()
                expert, n = ids.flatten()[pair].long(), outputs if form == "plain" else 2 * outputs
                sums, spread = torch.empty((count, n), dtype=torch.float64, device="cuda"), torch.empty((count, n), dtype=torch.float64, device="cuda")
                for e in range(experts):
                    m, we = expert == e, w[e, :n].double()
                    sums[m], spread[m] = rows_of_pairs[m] @ we.T, rows_of_pairs[m].abs() @ we.T.abs()
                factor = scale[pair].double()[:, None]
                want = (torch.nn.functional.silu(factor * sums[:, :outputs]) * (factor * sums[:, outputs:]) if form == "gated"
                        else sums.clamp(min=0) ** 2 if form == "plain" else sums)
        if form == "down":              # inner roundings of half a unit each at most
            assert bool(((got[64].double() - want).abs() <= inner * 2.0 ** -24 * spread).all())
        else:                           # the result's rounding to bfloat16 (2^-8, and as much again for the float steps in front of it)
            assert bool(((got[64].double() - want).abs() <= 2.0 ** -7 * want.abs() + 1e-5).all()), form
        assert got[128].shape[0] == count and torch.isfinite(got[128].float()).all() and torch.equal(got[64], got[128]), form
        assert torch.equal(got[16], got[64]) or (tokens == 131 and torch.allclose(got[16].float(), got[64].float(), rtol=2 ** -7, atol=1e-5)), form
