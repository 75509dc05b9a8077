"""Recurrences with a decay per row: the sums of a tile's queries and keys at the edges of the widths that the lanes take."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [31, 33, 63, 64, 65, 127, 128])
@pytest.mark.parametrize("tokens", [17, 32, 49, 150])
def test_rows_at_the_edges_of_the_lanes(N, tokens):
    """Against the recurrence token by token in 64 bits: portions that end in either tile of a piece, in pieces and in chunks, with decays
    down to zero.  A sum of up to ``tokens`` x N products in 32 bits, each product of up to ``tokens`` factors, is off by less than
    2 ** -24 x (tokens + log N + 8) of the sum of the products' sizes; the carried state goes over pieces, twice that."""
    from paged_llm_amd.csrc import ops
    H, P = 3, 40
    gen = torch.Generator().manual_seed(100 * N + tokens)
    q, k = (torch.randn(tokens, H, N, generator=gen) for _ in range(2))
    f = torch.sigmoid(torch.randn(tokens, H, N, generator=gen) * 3.0)
    f[torch.rand(tokens, H, N, generator=gen) < 0.02] = 0.0
    v = torch.randn(tokens, H, P, generator=gen)
    state = torch.randn(1, H * N * P, generator=gen)
    at = lambda *x: torch.tensor(x, dtype=torch.int32, device="cuda")
    st = state.cuda()
    y = ops.linear_recurrence(q.cuda(), k.cuda(), v.cuda(), None, st, 0, at(0), at(5), at(0, tokens), 1, max_q_len=tokens, row_decay=f.cuda())
    S = state.double().view(H, N, P)
    size, want, sizes = S.abs(), [], []
    for t in range(tokens):
        kv = k[t].double()[:, :, None] * v[t].double()[:, None, :]
        S, size = f[t].double()[:, :, None] * S + kv, f[t].double()[:, :, None] * size + kv.abs()
        want.append((S * q[t].double()[:, :, None]).sum(1))
        sizes.append((size * q[t].double().abs()[:, :, None]).sum(1))
    bound = 2.0 ** -23 * (tokens + N.bit_length() + 8)
    assert bool(((y.cpu().double().view(tokens, H, P) - torch.stack(want)).abs() <= bound * torch.stack(sizes)).all())
    assert bool(((st.cpu().double().view(H, N, P) - S).abs() <= bound * size).all())


@pytest.mark.parametrize("N", [64, 128])
def test_an_infinite_key_reaches_its_own_token_and_later_ones_only(N):
    from paged_llm_amd.csrc import ops
    q, k, f = torch.rand(32, 2, N) + 0.5, torch.rand(32, 2, N), torch.full((32, 2, N), 0.9)
    k[7, 1, N - 1] = float("inf")
    at = lambda *x: torch.tensor(x, dtype=torch.int32, device="cuda")
    y = ops.linear_recurrence(q.cuda(), k.cuda(), torch.rand(32, 2, 16).cuda() + 0.1, None, torch.zeros(1, 2 * N * 16, device="cuda"), 0, at(0), at(0),
                              at(0, 32), 1, max_q_len=32, row_decay=f.cuda()).cpu().view(32, 2, 16)
    assert bool(torch.isfinite(y[:, 0]).all() and torch.isfinite(y[:7, 1]).all() and not torch.isfinite(y[7:, 1]).any())


@pytest.mark.parametrize("N", [64, 128])
def test_neighbouring_rows_are_added_in_their_order(N, monkeypatch):
    """Sixteen lanes share a key, N / 16 neighbouring rows each: 2^24 + 1 + 1 - 2^24 is 0 in that order, and 1 where a lane had fewer rows."""
    from paged_llm_amd.csrc import ops
    monkeypatch.setattr(ops, "recurrence_form", lambda *a, **k: -1)             # (in pieces of 32 tokens, two tiles each)
    q, k, v = torch.zeros(32, 1, N), torch.ones(32, 1, N), torch.zeros(32, 1, 16)
    q[:, 0, :4] = torch.tensor([2.0 ** 24, 1.0, 1.0, -2.0 ** 24])
    v[0] = 1.0
    at = lambda *x: torch.tensor(x, dtype=torch.int32, device="cuda")
    y = ops.linear_recurrence(q.cuda(), k.cuda(), v.cuda(), None, torch.zeros(1, N * 16, device="cuda"), 0, at(0), at(0), at(0, 32), 1, max_q_len=32,
                              row_decay=torch.ones(32, 1, N).cuda())
    assert not bool(y[:16].any())


@pytest.mark.parametrize("N", [32, 64, 128])
@pytest.mark.parametrize("form", [-1, 64])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_a_gain_that_is_no_number_reaches_its_own_token_and_later_ones_only(N, form, value, monkeypatch):
    """In pieces and in chunks, with earlier tokens of the same tile, other tiles and another head beside it."""
    from paged_llm_amd.csrc import ops
    monkeypatch.setattr(ops, "recurrence_form", lambda *a, **k: form)
    q, k, v, gain = torch.rand(100, 2, N) + 0.1, torch.rand(100, 2, N), torch.rand(100, 2, 16) + 0.1, torch.rand(100, 2) + 0.1
    gain[41, 0] = value
    at = lambda *x: torch.tensor(x, dtype=torch.int32, device="cuda")
    y = ops.linear_recurrence(q.cuda(), k.cuda(), v.cuda(), None, torch.zeros(1, 2 * N * 16, device="cuda"), 0, at(0), at(0), at(0, 100), 1,
                              vscale=gain.cuda(), max_q_len=100, row_decay=torch.full((100, 2, N), 0.9).cuda()).cpu().view(100, 2, 16)
    assert bool(torch.isfinite(y[:, 1]).all() and torch.isfinite(y[:41, 0]).all()) and not bool(torch.isfinite(y[41:, 0]).any())
