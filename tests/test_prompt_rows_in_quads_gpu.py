"""Kernels of prompt rows that load four elements a thread, at the edges of what they hold."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("heads,dim,rot", [(1, 4, 0), (3, 8, 8), (5, 12, 8), (8, 256, 256), (7, 64, 24), (9, 132, 128)])
def test_rotations_by_quads_are_those_by_elements(heads, dim, rot, interleaved, dtype):
    """The same bits as by single elements, which rows one column on (off every boundary) still take."""
    from paged_llm_amd.csrc import ops
    gen = torch.Generator().manual_seed(dim)
    T, width = 37, heads * dim
    rows = torch.randn(T, 2 * width, generator=gen).to(dtype).cuda()
    off = torch.zeros(T, 2 * width + 4, dtype=dtype, device="cuda")
    off[:, 1:2 * width + 1] = rows
    positions = torch.randint(0, 50, (T,), generator=gen, dtype=torch.int32).cuda()
    angles = torch.rand(50, rot // 2, generator=gen) * 6.0
    tables = angles.cos().cuda(), angles.sin().cuda()
    args = (positions, *tables, heads, dim, rot, interleaved, 0.7)
    got = ops.rotary_to_float(rows, *args, second_at=width, scale2=0.3)
    assert torch.equal(got, ops.rotary_to_float(off[:, 1:], *args, second_at=width, scale2=0.3))
    x = rows.cpu().double().view(T, 2, heads, dim).transpose(0, 1)
    c, s = (t.cpu().double()[positions.cpu().long()][:, None] for t in tables)
    lo, hi = (x[..., 0:rot:2], x[..., 1:rot:2]) if interleaved else (x[..., :rot // 2], x[..., rot // 2:rot])
    turned = lo * c - hi * s, hi * c + lo * s
    want = x.clone()
    want[..., :rot] = torch.stack(turned, -1).flatten(-2) if interleaved else torch.cat(turned, -1)
    want *= torch.tensor([0.7, 0.3], dtype=torch.float64).view(2, 1, 1, 1)
    # (two products, their sum and the scale, each rounded to 24 bits)
    assert float((got.cpu().double() - want).abs().max()) <= 4 * 2.0 ** -24 * 2 * max(1.0, float(x.abs().max()))


@pytest.mark.parametrize("groups,group", [(4, 132), (5, 252), (4, 256), (6, 260), (4, 512), (7, 516), (4, 1024), (4, 1028), (5, 2048),
                                          (1, 1024), (1, 1040), (1, 8192), (2, 2056), (3, 300)])
@pytest.mark.parametrize("gate_first,act,weighted", [(True, "silu", True), (False, "sigmoid", False), (False, None, True)])
def test_norms_of_groups_at_the_edges_of_what_a_wavefront_holds(groups, group, gate_first, act, weighted):
    """Float rows against 64 bits: a sum of ``group`` squares in 32 bits is off by less than (64 + log2 group) x 2 ** -24 of itself here (a lane adds
    up to 32 in a row, half of which the root takes), the gate and the four products behind it by a few roundings more."""
    from paged_llm_amd.csrc import ops
    gen = torch.Generator().manual_seed(group)
    T, inner = 5, groups * group
    y, gate, w = torch.randn(T, inner, generator=gen) * 3, torch.randn(T, inner + 8, generator=gen), torch.rand(inner, generator=gen) + 0.5
    got = ops.gated_group_norm(y.cuda(), None if act is None else gate.cuda()[:, 4:4 + inner], w.cuda() if weighted else None, group, gate_first, 1e-5,
                               gate_activation=act, out_dtype=torch.float32).cpu().double()
    g = gate[:, 4:4 + inner].double()
    s = torch.ones_like(g) if act is None else torch.sigmoid(g) * (g if act == "silu" else 1.0)
    u = y.double() * s if gate_first else y.double()
    u = (u.view(T, groups, group) / (u.view(T, groups, group).square().mean(-1, keepdim=True) + 1e-5).sqrt()).view(T, inner)
    want = (u if gate_first else u * s) * (w.double() if weighted else 1.0)
    assert bool(((got - want).abs() <= 64 * 2.0 ** -24 * want.abs() + 1e-30).all())


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
