"""The matrix form of the linear recurrence: states of one tile and of sixteen, columns that fill no tile, portions of one token
more and less than a piece, one piece, many chunks, single tokens beside them, every kind of decay, rows of either type, strides
that wide loads cannot take, and values that are no numbers."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def ops():
    from paged_llm_amd.csrc import ops as o
    return o


def token_by_token(q, k, v, decay, S):
    """q, k [T, H, N], v [T, H, P] (the input factor in it), decay [T, H, N] in float64; outputs and the last state."""
    out = []
    for t in range(q.shape[0]):
        S = decay[t][:, :, None] * S + k[t][:, :, None] * v[t][:, None, :]
        out.append((q[t][:, None, :] @ S)[:, 0])
    return torch.stack(out), S


CASES = [  # heads, key heads, N, P, kind, type of rows, normaliser, columns of padding in the rows
    (2, 2, 16, 16, "head", torch.float32, False, 0), (4, 1, 128, 64, "steps", torch.bfloat16, False, 8), (2, 2, 256, 130, "constant", torch.float32, False, 0),
    (3, 3, 70, 66, "head", torch.float32, True, 3), (2, 2, 128, 256, "head", torch.float32, True, 0), (2, 2, 128, 128, "row", torch.float32, False, 0),
    (2, 2, 50, 30, "row", torch.float32, True, 1), (1, 1, 64, 200, "row", torch.float32, False, 4), (2, 1, 33, 17, "constant", torch.bfloat16, False, 5),
    (3, 3, 32, 32, "row", torch.bfloat16, False, 0), (2, 2, 20, 17, "row", torch.float32, True, 3), (2, 2, 32, 33, "row", torch.float32, False, 0)]


@pytest.mark.parametrize("chunk", [-1, 32, 96])
@pytest.mark.parametrize("H,KH,N,P,kind,dtype,normaliser,pad", CASES)
def test_pieces_against_token_by_token(H, KH, N, P, kind, dtype, normaliser, pad, chunk, monkeypatch):
    """Sequences that start and that go on, one without tokens, lengths around a piece and a chunk.  Bound: relative to the
    largest value 2e-5, forty times what float32 token by token shows against float64 at these sizes."""
    o = ops()
    monkeypatch.setattr(o, "recurrence_form", lambda *args: chunk)
    lens, starts = [33, 1, 0, 32, 131, 97], [0, 4, 0, 9, 0, 2]
    T, S_, ld = sum(lens), len(lens), P + 1 if normaliser else P
    g = torch.Generator().manual_seed(N + P)
    qk = torch.randn(T, 2 * KH * N + pad, generator=g).to(dtype)
    vv = torch.randn(T, H * P + pad, generator=g).to(dtype)
    q, k, v = qk[:, :KH * N].unflatten(1, (KH, N)), qk[:, KH * N:2 * KH * N].unflatten(1, (KH, N)), vv[:, pad:pad + H * P].unflatten(1, (H, P))
    state, slots = torch.randn(S_ + 1, H * N * ld + 5, generator=g), torch.tensor([5, 0, 2, 6, 1, 3], dtype=torch.int32)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    decay, vscale, skip, row, steps = None, None, None, None, None
    a = torch.rand(T, H, generator=g) * 0.9 + 0.1
    factor = torch.ones(T, H)
    if kind == "head":
        decay, vscale, skip = a, torch.rand(T, H, generator=g), torch.randn(H, generator=g)
        decay[7], factor = 0.0, vscale                           # (a decay of exactly 0 forgets everything)
    elif kind == "constant":
        decay = torch.linspace(0.9, 0.99, H)
        a = decay.expand(T, H)
    elif kind == "steps":
        raw, bias, a_log = torch.randn(T, H, generator=g).to(dtype), torch.randn(H, generator=g), torch.randn(H, generator=g)
        steps, skip = (raw, bias, a_log), torch.randn(H, generator=g)
        factor = torch.nn.functional.softplus(raw.double() + bias.double())
        a = torch.exp(-torch.exp(a_log.double()) * factor)
    else:
        row, vscale, skip = torch.rand(T, H, N, generator=g), torch.rand(T, H, generator=g), torch.randn(H, generator=g)
        row[:, :, ::3] *= 1e-3                                    # (rows that are forgotten within a few tokens)
        factor = vscale
    dev = lambda t: None if t is None else t.cuda()
    gq = dev(qk)
    st = dev(state.clone())
    y = o.linear_recurrence(gq[:, :KH * N].unflatten(1, (KH, N)), gq[:, KH * N:2 * KH * N].unflatten(1, (KH, N)), dev(vv)[:, pad:pad + H * P].unflatten(1, (H, P)),
                            dev(decay), st, 2, dev(slots), dev(torch.tensor(starts, dtype=torch.int32)), dev(cu), S_, vscale=dev(vscale), skip=dev(skip),
                            max_q_len=max(lens), step_sizes=None if steps is None else tuple(dev(t) for t in steps), normaliser=normaliser, row_decay=dev(row)).cpu()
    full = row.double() if row is not None else a.double()[:, :, None].expand(T, H, N)
    for s, n in enumerate(lens):
        lo, hi = int(cu[s]), int(cu[s + 1])
        before = state[slots[s], 2:2 + H * N * ld].double().view(H, N, ld) if starts[s] > 0 else torch.zeros(H, N, ld, dtype=torch.float64)
        after = st[slots[s], 2:2 + H * N * ld].cpu().double().view(H, N, ld)
        if n == 0:
            assert torch.equal(st[slots[s]].cpu(), state[slots[s]])
            continue
        many = lambda t: t[lo:hi].double().repeat_interleave(H // KH, dim=1)
        x = v[lo:hi].double()
        x1 = torch.cat([x, torch.ones(n, H, 1, dtype=torch.float64)], dim=2) if normaliser else x
        want, last = token_by_token(many(q), many(k), x1 * factor[lo:hi].double()[:, :, None], full[lo:hi], before)
        if skip is not None:
            want[:, :, :P] += skip.double()[:, None] * x
        got = y[lo:hi].double().view(n, H, ld)
        assert float((got - want).abs().max()) <= 2e-5 * float(want.abs().max()), s
        assert float((after - last).abs().max()) <= 2e-5 * float(last.abs().max()), s
    assert torch.equal(st[:, :2].cpu(), state[:, :2]) and torch.equal(st[:, 2 + H * N * ld:].cpu(), state[:, 2 + H * N * ld:]) and torch.equal(st[4].cpu(), state[4])


TALL = [(2, 1, 272, 20, "head", torch.float32, False, 0), (2, 2, 600, 70, "steps", torch.bfloat16, False, 8), (1, 1, 1024, 16, "constant", torch.float32, True, 3),
        (2, 2, 144, 40, "row", torch.float32, False, 4), (1, 1, 300, 66, "row", torch.bfloat16, True, 1)]


@pytest.mark.parametrize("chunk", [0, 16, 64])
@pytest.mark.parametrize("H,KH,N,P,kind,dtype,normaliser,pad", TALL)
def test_states_too_tall_for_pieces(H, KH, N, P, kind, dtype, normaliser, pad, chunk, monkeypatch):
    """More rows than the matrix form takes: token by token in one workgroup and in chunks, whose borders the lengths meet, pass and
    miss; the bound above (sums over up to 1,024 rows are cut into as many as there are wavefronts)."""
    assert ops().recurrence_form(131, 294, 6, H, N, P + normaliser, kind == "row", 256) == 16
    test_pieces_against_token_by_token(H, KH, N, P, kind, dtype, normaliser, pad, chunk, monkeypatch)


@pytest.mark.parametrize("by_row", [False, True])
@pytest.mark.parametrize("chunk", [-1, 64])
def test_a_value_that_is_no_number_reaches_later_tokens_only(by_row, chunk, monkeypatch):
    o = ops()
    monkeypatch.setattr(o, "recurrence_form", lambda *args: chunk)
    T, H, N, P = 70, 2, 48, 40
    g = torch.Generator().manual_seed(1)
    q, k, v, row = (torch.randn(T, H, n, generator=g).cuda() for n in (N, N, P, N))
    row, one = torch.sigmoid(row), torch.tensor([0], dtype=torch.int32, device="cuda")
    def run(v):
        state = torch.zeros(1, H * N * P, device="cuda")
        return o.linear_recurrence(q, k, v, None if by_row else torch.full((H,), 0.9, device="cuda"), state, 0, one, one,
                                   torch.tensor([0, T], dtype=torch.int32, device="cuda"), 1, max_q_len=T, row_decay=row if by_row else None).view(T, H, P)
    plain, bad = run(v), v.clone()
    bad[41, 1, 7] = float("inf")
    odd = run(bad)
    assert torch.equal(odd[:41], plain[:41]) and torch.equal(odd[:, 0], plain[:, 0])
    assert not bool(torch.isfinite(odd[41, 1, 7])) and not bool(torch.isfinite(odd[69, 1, 7]))
    keep = [c for c in range(P) if c != 7]
    assert torch.equal(odd[:, 1][:, keep], plain[:, 1][:, keep])


@pytest.mark.parametrize("H,KH,N,P,by_row", [(4, 2, 128, 64, False), (2, 2, 50, 30, True), (2, 1, 256, 20, False)])
def test_tokens_beside_a_short_portion_have_the_bits_they_have_alone(H, KH, N, P, by_row):
    """Below the bound that ``linear_recurrence`` states for chunks every token is the same whoever stands beside it: a portion of
    127 tokens, one of 20 and single tokens in one step, and each of the four token by token in steps of its own."""
    o = ops()
    lens, starts = [1, o.RECURRENCE_CHUNKS_FROM - 1, 1, 20], [3, 0, 1, 5]
    T, g = sum(lens), torch.Generator().manual_seed(N)
    q, k, v = (torch.randn(T, h, n, generator=g).cuda() for h, n in ((KH, N), (KH, N), (H, P)))
    decay, row = torch.rand(T, H, generator=g).cuda(), torch.rand(T, H, N, generator=g).cuda()
    state = torch.randn(4, H * N * P, generator=g).cuda()
    ints = lambda *x: torch.tensor(x, dtype=torch.int32, device="cuda")

    def step(st, slots, begun, lo, hi, cu):
        return o.linear_recurrence(q[lo:hi], k[lo:hi], v[lo:hi], None if by_row else decay[lo:hi], st, 0, slots, begun, ints(*cu), len(cu) - 1,
                                   max_q_len=max(b - a for a, b in zip(cu, cu[1:])), row_decay=row[lo:hi] if by_row else None)
    cu = [0, *torch.tensor(lens).cumsum(0).tolist()]
    together, alone = state.clone(), state.clone()
    y = step(together, ints(0, 1, 2, 3), ints(*starts), 0, T, cu)
    for s, n in enumerate(lens):
        for t in range(n):
            at = cu[s] + t
            assert torch.equal(step(alone, ints(s), ints(starts[s] + t), at, at + 1, [0, 1])[0], y[at]), (s, t)
    assert torch.equal(together, alone)


def test_which_form_a_step_takes():
    """Decode steps and portions of fewer than 128 tokens token by token, long prompts in chunks of whole pieces, longer portions beside
    many single tokens in pieces."""
    plan = ops().recurrence_form
    for n in (1, 64, 1024):
        assert plan(1, n, n, 64, 128, 64, False, 256) == 0
    for longest in (2, 16, 64, 127):
        for beside in (0, 1, 32):
            for heads, rows, columns, by_row in ((64, 128, 64, False), (8, 256, 512, False), (1, 16, 16, False), (16, 128, 128, True)):
                assert plan(longest, longest + beside, 1 + beside, heads, rows, columns, by_row, 256) == 0
    assert plan(100, 100, 1, 64, 128, 64, False, 256, chunks_from=17) == 32 and plan(64, 96, 33, 64, 128, 64, False, 256, chunks_from=17) == -1
    assert plan(16, 16, 1, 64, 128, 64, False, 256, chunks_from=17) == 0
    for tokens in (200, 2048, 8192):
        chunk = plan(tokens, tokens, 1, 8, 256, 512, False, 256)
        assert chunk > 0 and chunk % 32 == 0
    assert plan(128, 160, 33, 64, 128, 64, False, 256) == -1
    assert plan(4096, 4096, 1, 4, 512, 64, False, 256) in (64, 128) and plan(0, 5, 5, 4, 128, 64, False, 256) == 0
