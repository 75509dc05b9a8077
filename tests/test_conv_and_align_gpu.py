"""The convolution of long portions four channels a thread against the same channel by channel, and the sorting of (token, choice)
pairs by expert: pairs and experts around a wavefront and a workgroup."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def ops():
    from paged_llm_amd.csrc import ops as o
    return o


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("channels", [4, 1028])
@pytest.mark.parametrize("bias,activation", [(True, "silu"), (False, None)])
def test_four_channels_a_thread_give_the_same_bits(channels, bias, activation, dtype):
    """Rows that begin between two fours take the general kernel; the additions are the same."""
    o, g = ops(), torch.Generator().manual_seed(channels)
    lens, starts = [65, 1, 0, 257, 16, 2], [0, 3, 0, 7, 0, 5]
    T = sum(lens)
    x = torch.randn(T, channels, generator=g).to(dtype)
    w, b = torch.randn(channels, 4, generator=g).cuda(), torch.randn(channels, generator=g).cuda() if bias else None
    state = torch.randn(len(lens) + 1, 3 * channels + 2, generator=g).cuda()
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    where = (1, ints([3, 0, 6, 5, 1, 2]), ints(starts), ints([0, *torch.tensor(lens).cumsum(0).tolist()]), len(lens), max(lens))
    results = []
    for at, stride in ((4, channels + 8), (1, channels + 9)):
        rows = torch.zeros(T, stride, dtype=dtype)
        rows[:, at:at + channels] = x
        after = state.clone()
        results.append((o.causal_conv(rows.cuda()[:, at:at + channels], w, b, after, *where, activation=activation), after))
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])
    # against float64 for the first sequence, whose inputs before the first token are zeros: four products, rounded to the rows' type
    want = torch.nn.functional.conv1d(torch.nn.functional.pad(x[:65].double().T[None], (3, 0)), w.double().cpu()[:, None], b.double().cpu() if bias else None, groups=channels)[0].T
    want = torch.nn.functional.silu(want) if activation else want
    got = results[0][0][:65].double().cpu()
    assert (got - want).abs().max() <= (2 ** -8 if dtype == torch.bfloat16 else 2e-6) * want.abs().max()


@pytest.mark.parametrize("pairs,experts,extra", [(1, 1, 0), (1, 3, 2), (63, 64, 0), (64, 65, 1), (264, 8, 0), (1025, 1000, 24), (4096, 64, 8), (4097, 1024, 0), (9000, 7, 1)])
@pytest.mark.parametrize("tile_rows", [16, 128])
def test_pairs_sorted_by_expert(pairs, experts, extra, tile_rows):
    o, g = ops(), torch.Generator().manual_seed(pairs)
    ids = torch.randint(0, experts + extra, (pairs, 1), generator=g, dtype=torch.int32)
    if pairs > 100:
        ids[: pairs // 2] = experts // 2                          # (one expert with many tiles)
    sorted_pair, row_of_pair, tiles = (t.cpu() for t in o.moe_align(ids.cuda(), experts, tile_rows))
    flat = ids.flatten()
    kept = int((flat < experts).sum())
    assert torch.equal(flat[sorted_pair[:kept].long()], flat[flat < experts].sort().values)
    assert torch.equal(sorted_pair[:kept].sort().values, (flat < experts).nonzero().flatten().int())
    for p in range(pairs):
        assert row_of_pair[p] == -1 if flat[p] >= experts else sorted_pair[row_of_pair[p]] == p
    want, at = [], 0
    for e, rows in enumerate(torch.bincount(flat[flat < experts].long(), minlength=experts).tolist()):
        want += [[e, at + r, min(tile_rows, rows - r)] for r in range(0, rows, tile_rows)]
        at += rows
    assert tiles[: len(want)].tolist() == want and not bool(tiles[len(want):].any())
