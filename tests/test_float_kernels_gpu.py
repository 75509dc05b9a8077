"""The kernels of the true 32-bit path on the float matrix cores, at the edges of their tiles: products in every form of the
kernel."""

import pytest
import torch

from tests.test_kernels_gpu import rnd

pytestmark = pytest.mark.gpu


def ops():
    from paged_llm_amd.csrc import ops as o
    return o


@pytest.mark.parametrize("m,n,k", [(1, 16, 32), (17, 33, 31), (49, 65, 50), (65, 129, 513), (16, 64, 2047), (48, 64, 2048), (7, 70, 5632)])
def test_float_product_in_every_form(m, n, k):
    """Every tile gives the same bits.  Bound: a result is reached by at most ceil(K / 512) * 32 products in one chain, one
    addition of a pair and seven of the pairs, each rounded once (2^-24), so its error is at most that many roundings of the
    sum of the products' magnitudes."""
    o = ops()
    a, w = rnd(m, k, seed=1), rnd(n, k, seed=2)
    want, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    chain = -(-k // 512) * 32 + 8
    outs = []
    for tile in o.FLOAT_GEMM_TILES:
        for shift in (0, 1):                                    # rows that 16-byte loads can read, and rows that they cannot
            base_a, base_w = torch.zeros(m, k + 4 + shift), torch.zeros(n, k + 8 + shift)
            base_a[:, shift:k + shift], base_w[:, shift:k + shift] = a, w
            ga, gw, out = base_a.cuda()[:, shift:k + shift], base_w.cuda()[:, shift:k + shift], torch.full((m + 1, n), 7.0, device="cuda")
            code = o._fn("gemm_float.hip", "pllm_gemm_float")(ga.data_ptr(), ga.stride(0), 0, gw.data_ptr(), gw.stride(0), 0, out.data_ptr(), n, 0,
                                                              m, n, k, 1, *tile, o._stream())
            assert code == 0 and bool((out[m] == 7.0).all()), tile
            outs.append(out[:m].cpu())
    assert all(torch.equal(outs[0], x) for x in outs)
    assert bool(((outs[0].double() - want).abs() <= chain * 2.0 ** -24 * size + 1e-30).all())


def test_float_product_batches():
    """Heads side by side in the rows, one matrix each, written into wider rows."""
    o = ops()
    a, w = rnd(21, 5, 96, seed=3), rnd(5, 40, 96, seed=4)
    out = torch.zeros(21, 5, 43, device="cuda")
    o.gemm_heads(a.cuda(), o.HeadMatrices(w.cuda()), out=out[:, :, :40])
    want = torch.einsum("thk,hnk->thn", a.double(), w.double())
    assert float((out[:, :, :40].cpu().double() - want).abs().max() / want.abs().max()) <= 1e-6 and bool((out[:, :, 40:] == 0).all())
