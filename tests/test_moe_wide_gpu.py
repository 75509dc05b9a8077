"""The experts' products in wide tiles: the bits of the staged kernel, for every tile, at the edges of tiles, blocks and stages."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# one stage and more, fewer than and more than those under way; outputs past the last block of 16 and of a workgroup; experts without a row, with one
# and with several tiles; pairs handed past the experts; a factor on the pairs' rows
@pytest.mark.parametrize("tokens,top,experts,inner,outputs", [(3, 2, 3, 64, 4), (300, 2, 8, 128, 192), (517, 2, 3, 192, 328), (260, 4, 5, 320, 72), (131, 1, 1, 448, 2040)])
@pytest.mark.parametrize("form,activation", [("gated", "silu"), ("gated", "gelu_tanh"), ("plain", "gelu"), ("plain", "relu2"), ("down", "silu")])
def test_every_tile_gives_the_staged_bits(tokens, top, experts, inner, outputs, form, activation):
    from paged_llm_amd.csrc import ops
    gen = torch.Generator().manual_seed(tokens)
    h = torch.randn((tokens, inner), generator=gen).to(torch.bfloat16).cuda()
    w = (torch.randn((experts, (2 if form == "gated" else 1) * outputs, inner), generator=gen) * inner ** -0.5).to(torch.bfloat16).cuda()
    ids = torch.stack([torch.randperm(experts + 1, generator=gen)[:top] for _ in range(tokens)]).to(torch.int32).cuda()    # (expert `experts`: passed through)
    scale = torch.rand((tokens * top,), generator=gen).cuda() if form == "gated" else None
    pair_rows = torch.randn((tokens * top, inner), generator=gen).to(torch.bfloat16).cuda()

    def product(rows, columns):
        sorted_pair, row_of_pair, tiles = ops.moe_align(ids, experts, rows)
        place = row_of_pair.long()
        there = place >= 0
        if form == "down":
            x = torch.zeros_like(pair_rows)
            x[place[there]] = pair_rows[there]
            out = ops.moe_expert_gemm(x, w, tiles, sorted_pair, top, False, tile_rows=rows, wide_columns=columns)
        else:
            out = ops.moe_expert_gemm(h, w, tiles, sorted_pair, top, form == "gated", activation, tile_rows=rows, pair_scale=scale, plain=form == "plain",
                                      wide_columns=columns)
        return out[place[there]]
    want = product(64, 0)
    for rows in ops.MOE_WIDE_ROWS:
        for columns in ops.MOE_WIDE_COLUMNS:
            assert torch.equal(product(rows, columns), want), (rows, columns)


def test_plans():
    from paged_llm_amd.csrc import ops
    for case in ((2356, 8, 2048, 4096, False), (600, 8, 2048, 2048, True), (8192, 30, 2048, 1408, True), (1600, 16, 2048, 2048, False)):
        rows, first, down = ops.moe_wide_plan(*case, 256)
        assert rows in ops.MOE_WIDE_ROWS and first in ops.MOE_WIDE_COLUMNS and down in ops.MOE_WIDE_COLUMNS
    assert ops.moe_wide_plan(559, 8, 2048, 2048, True, 256) is None and ops.moe_wide_plan(4000, 16, 2048, 2016, False, 256) is None
    assert ops.moe_expected_tiles(80, 8, 64) == 8 and ops.moe_expected_tiles(2356, 8, 192) == 16
