"""Launch plans are plain functions of sizes; whatever they return must be something the kernels take."""

import numpy as np

from paged_llm_amd.csrc import ops


def test_attention_plan_always_returns_a_launch_the_kernels_take():
    rng = np.random.default_rng(7)
    lds = 160 * 1024
    for _ in range(3000):
        seqs = int(rng.choice([1, 2, 3, 7, 8, 16, 33, 64, 100, 256, 1000]))
        kv_heads = int(rng.choice([1, 2, 4, 8, 16]))
        group = int(rng.choice([1, 2, 3, 4, 5, 8, 16]))
        max_q = int(rng.choice([1, 1, 1, 2, 3, 8, 17, 64, 500]))
        max_k = max(max_q, int(rng.choice([1, 15, 64, 65, 200, 256, 1000, 2048, 2049, 8192, 100000])))
        d = int(rng.choice([16, 32, 48, 64, 80, 96, 112, 128, 160, 256]))
        waves, size, parts = ops.attention_plan(seqs, kv_heads, max_q, max_k, group, d, lds)
        what = f"plan({seqs}, {kv_heads}, {max_q}, {max_k}, {group}, {d}) = {(waves, size, parts)}"
        assert waves in (1, 4, 8), what
        assert size % 64 == 0 and size >= 0 and parts >= 1, what
        if size == 0:
            assert parts == 1, what
        else:
            assert parts > 1 and (parts - 1) * size < max_k <= parts * size, what     # the partitions cover the keys, none is empty
            assert kv_heads * parts <= 65535, what                                  # a grid dimension
        if max_q * group > 64:
            assert (waves, size, parts) == (1, 0, 1), what                          # prompt portions: the other kernel
        if waves > 1:
            ncb = 1 if max_q * group <= 16 else (2 if max_q * group <= 32 else 4)
            assert ops._merge_lds_bytes(ncb, waves, d) <= lds, what


def test_attention_plan_of_up_to_512_keys_in_one_piece():
    """Eight wavefronts take 257 to 512 keys of up to 16 columns without a merge, for heads up to 128 and work items that fit the compute
    units; every edge of that has another plan beyond it."""
    plan, lds = ops.attention_plan, 160 * 1024
    for keys in (257, 300, 512):
        assert plan(1, 4, 1, keys, 8, 64, lds) == plan(8, 4, 1, keys, 16, 128, lds) == plan(64, 4, 1, keys, 1, 64, lds) == (8, 0, 1)
    assert plan(1, 4, 1, 256, 8, 64, lds) == (4, 0, 1) and plan(1, 4, 1, 513, 8, 64, lds) == (4, 256, 3)
    assert plan(1, 4, 1, 512, 17, 64, lds) == (4, 256, 2) and plan(1, 4, 2, 512, 8, 64, lds) == (8, 0, 1) and plan(1, 4, 3, 512, 8, 64, lds) == (4, 256, 2)
    assert plan(1, 4, 1, 512, 8, 144, lds) == (4, 256, 2) and plan(257, 1, 1, 512, 8, 64, lds) == (4, 0, 1)
    rng = np.random.default_rng(8)
    for _ in range(300):
        seqs, kv_heads, group = int(rng.integers(1, 300)), int(rng.choice([1, 2, 4, 8, 16])), int(rng.choice([1, 3, 8, 16]))
        keys, d = int(rng.choice([257, 300, 511, 512])), int(rng.choice([16, 48, 64, 96, 128, 160]))
        waves, size, parts = plan(seqs, kv_heads, 1, keys, group, d, lds)
        assert waves in (4, 8) and ((size, parts) == (0, 1) or (parts > 1 and (parts - 1) * size < keys <= parts * size))
        assert ops._merge_lds_bytes(1, waves, d) <= lds


def test_attention_plan_depends_on_sizes_only():
    a = ops.attention_plan(8, 4, 1, 2048, 8, 64, 160 * 1024)
    assert a == ops.attention_plan(8, 4, 1, 2048, 8, 64, 160 * 1024) == (4, 256, 8)


def test_graph_batch_sizes_cover_every_batch_with_at_most_half_as_many_rows_again():
    from paged_llm_amd.engine.runner import ModelRunner
    sizes = [ModelRunner._bucket(n) for n in range(1, 600)]
    assert all(b >= n and 2 * b <= 3 * n + 1 for n, b in zip(range(1, 600), sizes))      # never fewer rows, at most half again
    assert sizes == sorted(sizes)
    assert len(set(sizes)) <= 24                                                       # few graphs for a batch that shrinks one by one
    assert [ModelRunner._bucket(n) for n in (1, 2, 3, 4, 5, 6, 7, 8, 9, 13, 64, 65)] == [1, 2, 3, 4, 6, 6, 8, 8, 12, 16, 64, 96]


def test_ranges_of_the_inner_dimension_are_never_empty():
    """The products' plans cut K into ranges of equal numbers of stages; whatever the sizes, no range is left empty
    (a matrix of 2048 x 5632 at 150 rows once asked for 16 ranges of 6 of its 88 stages)."""
    from paged_llm_amd.csrc import ops
    for rows in (17, 64, 100, 128, 129, 150, 160, 161, 264, 320, 400, 512, 640):
        for n, k in ((2048, 2048), (2048, 5632), (2560, 2048), (4096, 4096), (96, 992), (2048, 14336), (32, 32)):
            for cus in (256, 304, 64):
                ranges, stages = ops.tile_linear_plan(rows, n, k, cus), -(-k // 64)
                assert ranges == 1 or -(-stages // ranges) * (ranges - 1) < stages, (rows, n, k, ranges)
                _, ranges = ops.stream_linear_plan(rows, n, k, cus)
                stages = -(-k // 256)
                assert ranges == 1 or -(-stages // ranges) * (ranges - 1) < stages, (rows, n, k, ranges)


def test_streaming_product_plans_by_sizes():
    from paged_llm_amd.csrc import ops
    plan, cus = ops.stream_linear_plan, 256
    assert plan(64, 2048, 5632, cus) == (2, 4)                # 64 blocks of 32 weight rows x 4 ranges: a workgroup per compute unit
    assert plan(64, 2048, 2048, cus) == (2, 4) and plan(64, 2560, 2048, cus) == (2, 3)
    assert plan(64, 4096, 14336, cus) == (4, 4)               # long K, few rows: four blocks, fewer reads of the rows
    assert plan(128, 4096, 14336, cus) == (2, 2)
    assert plan(64, 2048, 2048, cus, partial=False) == (1, 1) and plan(64, 6144, 4096, cus, partial=False) == (2, 1)
    assert ops.gated_blocks_per_workgroup(5632, cus) == 3 and ops.gated_blocks_per_workgroup(14336, cus) == 4
    assert ops.gated_blocks_per_workgroup(8192, cus) == 4     # 1024 blocks: 342 workgroups of three would need a second round


def test_tiles_of_the_experts_products_by_sizes():
    import torch
    from paged_llm_amd.csrc import ops
    rows = lambda tokens, top, experts, width, ff, dtype=torch.bfloat16: ops.moe_tile_rows(tokens * top, experts, dtype, width, ff, width)
    assert rows(64, 4, 16, 2048, 2048) == 16 and rows(127, 4, 16, 2048, 2048) == 16      # fewer than 32 pairs an expert
    assert rows(128, 4, 16, 2048, 2048) == 128 and rows(2048, 4, 16, 1024, 1024) == 128
    assert rows(256, 4, 16, 1024, 1024) == 64 and rows(512, 4, 16, 1024, 1024) == 128    # small experts: tiles that reach every compute unit
    assert rows(2048, 4, 16, 2048, 2048, torch.float32) == 16 and rows(2048, 4, 16, 50, 2048) == 16      # the plain kernel's tiles


def test_decode_attention_of_large_heads_keeps_to_four_wavefronts():
    for d in (144, 160, 256):
        assert ops.attention_plan(64, 1, 1, 2048, 16, d, 160 * 1024) == (4, 512, 4)
    assert ops.attention_plan(64, 1, 1, 2048, 16, 128, 160 * 1024) == (8, 512, 4)


def test_float_products_of_short_rows_take_small_tiles_until_the_gpu_is_full():
    """What a workgroup takes whatever its columns counts: few rows of heads with short rows go in the smallest tiles, large steps in large
    ones, and products of long rows as the rounds say."""
    plan = ops.float_gemm_plan
    for rows in (1, 8, 16):
        for heads in (1, 16, 64):
            assert plan(rows, 64, 64, heads, 256) == (1, 1)
    assert plan(130, 128, 64, 16, 256) in ((1, 2), (2, 2)) and plan(4096, 64, 64, 64, 256) == (4, 4)
    assert plan(301, 2048, 2048, 1, 256) == (3, 4) and plan(301, 2560, 2048, 1, 256) == (4, 4) and plan(8, 2048, 2048, 1, 256) == (1, 1)
    assert plan(1500, 64, 64, 64, 256) == plan(777, 128, 128, 16, 256) == (2, 2) and plan(2048, 256, 256, 16, 256) == (3, 4)
    assert plan(8, 32000, 2048, 1, 256) == plan(1, 32000, 2048, 1, 256) == (1, 1) and plan(4096, 2048, 5632, 1, 256) == (4, 4)


def test_recurrences_with_a_decay_per_row_run_in_chunks_beside_few_single_tokens():
    """Pieces, one workgroup a sequence and head, are for portions beside so many single tokens that a workspace of all their states costs more."""
    plan = ops.recurrence_form
    assert plan(2048, 2080, 33, 64, 64, 64, True, 256) > 0 and plan(130, 138, 9, 16, 128, 128, True, 256) > 0
    assert plan(130, 162, 33, 4, 32, 32, True, 256) == 32 and plan(700, 1164, 6, 64, 64, 64, True, 256) > 0
    assert plan(8192, 8192, 1, 64, 64, 64, True, 256) <= 1024
    assert plan(500, 564, 65, 16, 128, 128, True, 256) == -1 and plan(500, 564, 65, 100, 32, 32, True, 256) == -1


def test_pieces_of_tall_states_come_in_whole_rounds():
    """Nine sequences of 8 heads of 256 x 512 are 288 workgroups of eight wavefronts: two rounds of pieces, longer than 17 tokens one by one."""
    plan = ops.recurrence_form
    assert plan(17, 25, 9, 8, 256, 512, False, 256, chunks_from=17) == 0 and plan(17, 24, 8, 8, 256, 512, False, 256, chunks_from=17) == -1
    assert plan(100, 108, 9, 8, 256, 512, False, 256, chunks_from=17) == -1


def test_float32_steps_keep_the_order_of_their_recurrences_below_the_stated_bound():
    from types import SimpleNamespace

    import torch

    from paged_llm_amd.parts.recurrent import _chunks_from
    assert _chunks_from(SimpleNamespace(dtype=torch.float32)) == ops.RECURRENCE_CHUNKS_FROM == 128
    assert _chunks_from(SimpleNamespace(dtype=torch.bfloat16)) == 17           # (steps of up to 16 rows keep their products' order as well)


def test_wide_products_fill_one_round():
    """One round of workgroups, half of the compute units busy at least; each tile's share of them and its longest K, with what lies just past them."""
    plan, BF, F, G = ops.wide_linear_plan, ops.SL_BF16, ops.SL_F32, ops.SL_GATED
    assert plan(264, 2048, 2048, BF, 256) == (64, 64) and plan(200, 1024, 2048, BF, 256) is None and plan(192, 6144, 2048, F, 256) == (64, 128) and plan(1280, 2592, 2048, F, 256) == (128, 128)
    assert plan(256, 2048, 3072, BF, 256) == (64, 64) and plan(256, 2048, 4096, BF, 256) is None and plan(320, 2048, 4096, BF, 256) == (64, 64)
    assert plan(512, 2048, 6144, BF, 256) is None and plan(512, 2048, 6144, F, 256) == (64, 64) and plan(512, 2048, 8192, F, 256) == (64, 64) and plan(512, 2048, 8256, F, 256) is None
    assert plan(192, 4096, 14336, BF, 256) == (64, 64) and plan(256, 4096, 14336, BF, 256) is None
    assert plan(896, 2048, 8192, F, 256) == (96, 96) and plan(768, 2048, 2048, BF, 256) is None and plan(768, 2048, 1536, BF, 256) == (64, 128) and plan(512, 2560, 2048, BF, 256) == (96, 96)
    assert plan(256, 8192, 2048, BF, 256) == (64, 128) and plan(512, 4096, 4096, BF, 256) == (64, 128) and plan(512, 4096, 8192, BF, 256) == (80, 128)
    assert plan(1280, 2048, 8192, BF, 256) == (80, 128) and plan(1536, 2048, 5632, BF, 256) == (96, 128) and plan(1536, 2048, 8192, BF, 256) is None
    assert plan(2048, 2048, 4096, BF, 256) == (128, 128) and plan(2048, 2048, 4608, BF, 256) is None and plan(1536, 3072, 3072, BF, 256) == (128, 160)
    assert plan(2048, 8192, 2048, BF, 256) is None and plan(2048, 2560, 2048, ops.SL_ROPE_KV, 256) == (128, 160)
    assert plan(256, 8192, 1024, G, 256) == (64, 128) and plan(192, 8192, 1024, G, 256) is None and plan(320, 4096, 2048, G, 256) is None
    assert plan(768, 1536, 1024, G, 256) == (64, 128) and plan(448, 2560, 2048, G, 256) == (96, 96) and plan(384, 3072, 3072, G, 256) == (96, 96) and plan(384, 3072, 4096, G, 256) is None
    assert plan(448, 11264, 2048, G, 256) == (192, 192) and plan(640, 8192, 2048, G, 256) is None and plan(768, 8192, 1024, G, 256) == (192, 192)
    assert plan(777, 11264, 2048, G, 256) == (160, 256) and plan(896, 11264, 2048, G, 256) == (224, 192) and plan(1024, 11264, 2048, G, 256) == (256, 192)
    assert plan(512, 16384, 2048, G, 256) is None and plan(576, 16384, 2048, G, 256) == (160, 256)
    assert plan(2048, 11264, 2048, G, 256) is None and plan(777, 2048, 2080, BF, 256) is None and plan(777, 2046, 2048, BF, 256) is None
    for rows in (129, 500, 2000, 8192):
        for weight_rows in (64, 1000, 2560, 11264, 28672):
            for epi in (ops.SL_BF16, ops.SL_F32, ops.SL_ROPE_KV, ops.SL_GATED):
                tile = plan(rows, weight_rows, 2048, epi, 256)
                if tile is not None:
                    assert 128 <= -(-rows // tile[0]) * -(-weight_rows // tile[1]) <= 256


def test_gated_products_take_the_tile_of_the_least_estimate():
    """From 129 rows and K = 1024 on, whatever the rounds; None where the tiled kernel's own tiles fill a round, for short K, and past 32-bit offsets."""
    plan = ops.wide_gated_plan
    assert plan(2048, 11264, 2048, 256) == (256, 352) and plan(1024, 16384, 2048, 256) == (256, 256) and plan(777, 11264, 2048, 256) == (160, 256)
    assert plan(264, 28672, 4096, 256) == (288, 128) and plan(200, 16384, 2048, 256) == (128, 128) and plan(200, 4096, 1024, 256) == (64, 64)
    assert plan(264, 16384, 2048, 256) is None and plan(160, 28672, 4096, 256) is None and plan(2048, 11264, 960, 256) is None
    assert plan(2048, 11264, 2080, 256) is None and plan(2048, 11260, 2048, 256) is None and plan(1 << 17, 8192, 1024, 256) is None
    for rows in (129, 161, 257, 500, 2000, 8192):
        for weight_rows in (64, 1000, 2560, 11264, 28672):
            tile = plan(rows, weight_rows, 2048, 256)
            assert tile is None or tile in ops.WIDE_TILES + ops.WIDE_LARGE_TILES


def test_plain_products_take_large_tiles_where_square_ones_begin_a_round():
    """One round of 256 x 288 to 256 x 352 where 256 x 256 needs two, and so on; None in front of and behind that, for short K, and past 32-bit offsets."""
    plan = ops.wide_plain_plan
    assert plan(2048, 8512, 2048, 256) == (256, 288) and plan(2048, 8192, 2048, 256) is None and plan(2048, 10240, 1024, 256) == (256, 320)
    assert plan(1777, 12288, 2048, 256) == (256, 352) and plan(2048, 12288, 2048, 256) is None and plan(1178, 32000, 2048, 256) == (256, 320)
    assert plan(640, 32000, 2048, 256) == (320, 256) and plan(512, 32000, 2048, 256) is None and plan(777, 2048, 5632, 256) is None
    assert plan(2048, 8512, 960, 256) is None and plan(2048, 8512, 2080, 256) is None and plan(2048, 8510, 2048, 256) is None and plan(70000, 8512, 2048, 256) is None
    assert plan(2048, 8512, 1 << 21, 256) is None and ops.wide_gated_plan(2048, 11264, 1 << 21, 256) is None


def test_sigmoid_attention_counts_the_columns_that_there_are():
    """More wavefronts a tile where tiles are few; padding and short sequences beside a long one no longer count as long ones."""
    plan = ops.sigmoid_attention_plan
    assert plan(8, 64, 100) == plan(8, 64, 100, 800) == (1, 8, False)
    assert plan(896 * 8, 64, 2 * 4) == (2, 1, False) and plan(896 * 8, 64, 2 * 4, 896 * 32) == (2, 4, False)
    assert [plan(8 * t, 64, 4, 32 * t)[:2] for t in (64, 65, 384, 385, 960, 961, 1536, 1537)] == [(1, 8), (1, 4), (1, 4), (2, 4), (2, 4), (2, 2), (2, 2), (2, 1)]
    assert plan(4 * 700, 128, 4, 16 * 700) == (1, 2, False) and plan(40, 256, 1, 40) == (1, 4, False)


def test_experts_stay_with_the_staged_kernel_where_wide_tiles_were_behind():
    """Small experts of few rows (600 tokens with 8 of 64 of 512: 61 us staged, 86 in the wide tiles once chosen; of 1,536 at width 4,096 511 and 632)."""
    for case in ((4800, 64, 1024, 512, True), (4800, 64, 4096, 1536, True)):
        assert ops.moe_wide_plan(*case, 256) is None, case
    for case in ((4096, 16, 2048, 2048, False), (2048, 8, 2048, 4096, False), (4096, 8, 2048, 2048, True), (1600, 16, 2048, 2048, False)):
        rows, first, down = ops.moe_wide_plan(*case, 256)
        assert rows in ops.MOE_WIDE_ROWS and first in ops.MOE_WIDE_COLUMNS and down in ops.MOE_WIDE_COLUMNS


def test_sequences_behind_a_window_are_taken_as_they_come():
    """The order by length is for layers that see whole sequences: without a window, or with one that no sequence is longer than."""
    assert ops.longest_in_turn(0, 2000) == ops.longest_in_turn(2000, 2000) == ops.longest_in_turn(-4096, 2000) == 2000
    for window in (1, 128, 512, 1024, 1999, -512):
        assert ops.longest_in_turn(window, 2000) == 0
    assert ops.longest_in_turn(0, 0) == ops.longest_in_turn(512, 0) == 0
