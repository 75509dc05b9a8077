"""The selective scan in chunks, whose rows are asked for ahead: portions around every remainder of the tokens asked for at once."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [8, 16, 32, 64])
@pytest.mark.parametrize("lens", [[257], [258, 1], [261, 0, 2], [263], [300, 31], [512]])
def test_portions_around_the_tokens_asked_for_at_once(lens, N):
    """Against the scan in 64 bits.  A result is a sum of N x tokens products, each behind a decay whose exponent is a sum of up to ``tokens``
    steps in 32 bits: off by less than 4 x 2 ** -24 x (tokens + 64) of the sum of the products' sizes."""
    from paged_llm_amd.csrc import ops
    gen = torch.Generator().manual_seed(sum(lens) + N)
    T, S, C = sum(lens), len(lens), 100
    rand = lambda *shape: torch.randn(*shape, generator=gen)
    x, z, raw, bias, bc, skip, state = rand(T, C), rand(T, C), rand(T, C), rand(C) - 3.0, rand(T, 2 * N), rand(C), rand(S, N * C)
    a2 = -torch.rand(N, C, generator=gen) * 4.0
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    cu, starts, held = [sum(lens[:s]) for s in range(S + 1)], [(s + 1) % 2 for s in range(S)], state.cuda()
    y = ops.selective_scan(x.cuda(), raw.cuda(), bias.cuda(), bc.cuda(), a2.cuda(), skip.cuda(), z.cuda(), held, i32(list(range(S))), i32(starts), i32(cu), S,
                           max(lens)).cpu().double()
    bound = 4 * 2.0 ** -24 * (max(lens) + 64)
    dt = torch.nn.functional.softplus(raw.double() + bias.double())
    for s in range(S):
        h = state[s].double().view(N, C) * starts[s]
        size = h.abs()
        for t in range(cu[s], cu[s + 1]):
            decay, dx = torch.exp2(a2.double() * dt[t]), (dt[t] * x[t].double()) * bc[t, :N].double()[:, None]
            h, size = decay * h + dx, decay * size + dx.abs()
            gate, c = torch.nn.functional.silu(z[t].double()), bc[t, N:].double()[:, None]
            want = ((h * c).sum(0) + skip.double() * x[t].double()) * gate
            most = ((size * c.abs()).sum(0) + (skip * x[t]).abs().double()) * gate.abs()
            assert bool(((y[t] - want).abs() <= bound * most + 1e-12).all()), (s, t)
        if lens[s]:
            assert bool(((held[s].cpu().double().view(N, C) - h).abs() <= bound * size + 1e-12).all())
        else:
            assert torch.equal(held[s].cpu(), state[s])


@pytest.mark.parametrize("N", [32, 64, 256])
def test_launches_of_many_wavefronts_give_the_bits_of_few(N):
    """Beyond three wavefronts a SIMD states of more than 16 numbers a lane do not ask for rows ahead: the first channels alone, which do, are the same."""
    from paged_llm_amd.csrc import ops
    gen = torch.Generator(device="cuda").manual_seed(N)
    T, C, few = 2048, 4096, 70
    rand = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")
    x, z, raw, bias, bc, skip, state = rand(T, C), rand(T, C), rand(T, C), rand(C) - 3.0, rand(T, 2 * N), rand(C), rand(1, N * C)
    a2 = -torch.rand(N, C, generator=gen, device="cuda") * 4.0
    at = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")

    def scan(c):
        held = state.view(N, C)[:, :c].reshape(1, -1).clone()
        part = lambda t: t[..., :c].contiguous()
        y = ops.selective_scan(part(x), part(raw), part(bias), bc, part(a2), part(skip), part(z), held, at(0), at(1), at(0, T), 1, T)
        return y, held.view(N, c)
    for whole, first in zip(scan(C), scan(few)):
        assert torch.equal(whole[:, :few], first)
