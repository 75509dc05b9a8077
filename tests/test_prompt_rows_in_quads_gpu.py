"""Kernels of prompt rows that load four elements a thread, at the edges of what they hold."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("lens", [[256, 0], [257, 1, 2, 3], [0, 300], [2, 263, 0, 0], [1, 1, 1, 1, 1, 255 + 9]])
def test_convolutions_of_long_portions_beside_short_and_empty_ones(lens, dtype):
    """Carried and fresh states beside every length below the taps: outputs and what is left, against 64 bits."""
    from paged_llm_amd.csrc import ops
    gen = torch.Generator().manual_seed(sum(lens))
    C, S, T = 1028, len(lens), sum(lens)
    x, w, b = torch.randn(T, C, generator=gen).to(dtype), torch.randn(C, 4, generator=gen), torch.randn(C, generator=gen)
    for turn in range(2):
        starts = [(s + turn) % 2 * 4 for s in range(S)]
        state = torch.randn(S + 1, C * 3, generator=gen)
        held = state.clone().cuda()
        i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
        cu = [sum(lens[:s]) for s in range(S + 1)]
        y = ops.causal_conv(x.cuda(), w.cuda(), b.cuda(), held, 0, i32(list(range(S))[::-1]), i32(starts), i32(cu), S, max(lens), activation=None).cpu().double()
        for s in range(S):
            slot = S - 1 - s
            before = state[slot].view(C, 3) if starts[s] else torch.zeros(C, 3)
            rows = torch.cat([before.double(), x[cu[s]:cu[s + 1]].double().T], 1)
            assert torch.equal(held[slot].cpu().view(C, 3).double(), rows[:, rows.shape[1] - 3:])
            if lens[s]:
                parts = rows.unfold(1, 4, 1) * w.double()[:, None]
                want, size = (parts.sum(-1) + b.double()[:, None]).T, (parts.abs().sum(-1) + b.double().abs()[:, None]).T
                # (four fused additions; bfloat16 rounds the result to eight bits)
                bound = 5 * 2.0 ** -24 * size + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0.0)
                assert bool(((y[cu[s]:cu[s + 1]] - want).abs() <= bound).all())
        assert torch.equal(held[S].cpu(), state[S])
