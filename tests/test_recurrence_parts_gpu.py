"""The recurrence with one decay per head as products of bfloat16 parts: rows of every pair of types, portions around a piece of 32 and
64 tokens, strides that wide loads cannot take, queries and keys that are no numbers, and values too large for bfloat16."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def ops():
    from paged_llm_amd.csrc import ops as o
    return o


def run(o, q, k, v, decay, T, normaliser=False, skip=None):
    H, N, P = v.shape[1], q.shape[2], v.shape[2] + normaliser
    one = torch.zeros(1, dtype=torch.int32, device="cuda")
    state = torch.zeros(1, H * N * P, device="cuda")
    y = o.linear_recurrence(q, k, v, decay, state, 0, one, one, torch.tensor([0, T], dtype=torch.int32, device="cuda"), 1, max_q_len=T,
                            normaliser=normaliser, skip=skip).view(T, H, P)
    return y, state.view(H, N, P)


def oracle(q, k, v, decay, normaliser=False, skip=None):
    q, k, v, decay = (x.double().cpu() for x in (q, k, v, decay))
    H, KH = v.shape[1], q.shape[1]
    q, k = (x.repeat_interleave(H // KH, 1) for x in (q, k))
    vv = torch.cat([v, torch.ones_like(v[..., :1])], -1) if normaliser else v
    S, out = torch.zeros(H, q.shape[2], vv.shape[2], dtype=torch.float64), []
    for t in range(q.shape[0]):
        S = decay[t][:, None, None] * S + k[t][:, :, None] * vv[t][:, None, :]
        out.append((q[t][:, None, :] @ S)[:, 0])
        if skip is not None:
            out[-1][:, :v.shape[2]] += skip.double().cpu()[:, None] * v[t]
    return torch.stack(out), S


@pytest.mark.parametrize("chunk", [-1, 64, 96])
@pytest.mark.parametrize("q_type,v_type", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.bfloat16), (torch.float32, torch.float32), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("H,KH,N,P,normaliser", [(2, 1, 128, 64, False), (2, 2, 63, 66, True), (1, 1, 200, 131, False), (2, 1, 8, 8, True)])
def test_types_and_lengths_around_a_piece(H, KH, N, P, normaliser, q_type, v_type, chunk, monkeypatch):
    """Bound: the largest difference over the largest value 4e-6: a sum of up to N + T products of float parts, each rounded to 2^-24,
    shows about sqrt(N + T) 2^-24 = 1e-6 (token by token 1.5e-6 was measured)."""
    o = ops()
    monkeypatch.setattr(o, "recurrence_form", lambda *args: chunk)
    g = torch.Generator().manual_seed(N + P)
    for T in (31, 33, 63, 65, 130):
        q, k, v = (torch.randn(T, h, n, generator=g).to(t).cuda() for h, n, t in ((KH, N, q_type), (KH, N, q_type), (H, P, v_type)))
        decay, skip = (0.7 + 0.3 * torch.rand(T, H, generator=g)).cuda(), torch.randn(H, generator=g).cuda()
        y, S = run(o, q, k, v, decay, T, normaliser, skip)
        want_y, want_S = oracle(q, k, v, decay, normaliser, skip)
        for got, want in ((y, want_y), (S, want_S)):
            assert (got.double().cpu() - want).abs().max() <= 4e-6 * want.abs().max(), (T, N, P)


@pytest.mark.parametrize("chunk", [-1, 64])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("which,value", [("k", float("inf")), ("q", float("-inf")), ("q", float("nan")), ("k", float("nan")), ("v", 3.4e38), ("v", float("nan"))])
def test_what_is_no_number_stays_where_it_belongs(which, value, dtype, chunk, monkeypatch):
    """Tokens in front and the other head have the bits that they have without it; where a token-by-token sum is infinite or no
    number, so is the result, with the same sign.  (3.4e38 is a float that rounds to no bfloat16 number.)"""
    o = ops()
    T, H, N, P, at = 90, 2, 40, 36, 37
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(T, H, n, generator=g).to(dtype).cuda() for n in (N, N, P))
    decay = torch.full((T, H), 0.9, device="cuda")
    bad = {"q": q, "k": k, "v": v}
    bad[which] = bad[which].clone()
    bad[which][at, 1, 5] = value
    monkeypatch.setattr(o, "recurrence_form", lambda *args: chunk)
    plain, (odd, odd_state) = run(o, q, k, v, decay, T)[0], run(o, bad["q"], bad["k"], bad["v"], decay, T)
    monkeypatch.setattr(o, "recurrence_form", lambda *args: 0)
    want, want_state = run(o, bad["q"], bad["k"], bad["v"], decay, T)
    assert torch.equal(odd[:at], plain[:at]) and torch.equal(odd[:, 0], plain[:, 0])
    for got, ref in ((odd, want), (odd_state, want_state)):
        fine = torch.isfinite(ref)
        assert torch.equal(torch.isfinite(got), fine) and torch.equal(torch.isnan(got), torch.isnan(ref))
        assert torch.equal(got[~fine & ~torch.isnan(ref)], ref[~fine & ~torch.isnan(ref)])
        small = fine & (ref.abs() < 1e6)
        assert (got[small] - ref[small]).abs().max() <= 1e-4 * ref[small].abs().max()


def test_pieces_of_bfloat16_rows_are_longer():
    """Portions of up to 100 tokens and those beside single tokens in pieces, longer ones in chunks of whole pieces of 64."""
    o = ops()
    def plan(*args):
        return o.recurrence_form(*args, 256, 17, o.RECURRENCE_LONG_PIECE)
    assert plan(100, 100, 1, 64, 128, 64, False) == -1 and plan(2048, 2080, 33, 64, 128, 64, False) == -1
    assert plan(200, 200, 1, 64, 128, 64, False) == 64 and plan(2048, 2048, 1, 64, 128, 64, False) == 256 and plan(777, 777, 1, 64, 128, 64, False) == 128
    for T in (129, 300, 3000):
        form = plan(T, T, 1, 8, 128, 257, False)
        assert form > 0 and form % 64 == 0
    assert plan(200, 200, 1, 8, 256, 512, False) == 32
