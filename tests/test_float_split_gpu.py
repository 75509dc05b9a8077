"""Float products whose weights come as their bfloat16 parts, laid out once: the bits of the products that split the floats themselves."""

import pytest
import torch

from tests.test_kernels_gpu import rnd

pytestmark = pytest.mark.gpu


def ops():
    from paged_llm_amd.csrc import ops as o
    return o


def each_tile(monkeypatch):
    for tile in ops().FLOAT_SPLIT_TILES:
        monkeypatch.setattr(ops(), "float_split_plan", lambda *a, tile=tile: tile)
        yield tile


# rows and weight rows past the last tile, one step of columns, slices without columns (K = 520, 1408), an odd number of steps a slice, a tail
@pytest.mark.parametrize("m,n,k", [(1, 16, 32), (33, 70, 520), (96, 130, 1408), (65, 2048, 2052), (150, 48, 3000), (70, 2049, 512)])
def test_plain_product_from_parts(m, n, k, monkeypatch):
    o = ops()
    a, w = rnd(m, k, seed=1).cuda(), rnd(n, k, seed=2).cuda()
    want, split = o.gemm_generic(a, w), o.float_split_weights(w)
    for tile in each_tile(monkeypatch):
        assert torch.equal(o.gemm_float_split(a, w, split), want), tile


@pytest.mark.parametrize("m,ff,k", [(40, 129, 512), (97, 12, 100), (130, 40, 2048)])
def test_gated_product_from_parts(m, ff, k, monkeypatch):
    o = ops()
    a, w = rnd(m, k, seed=3).cuda(), rnd(2 * ff, k, seed=4).cuda()
    want, split = o.gemm_float_gated(a, w), o.float_split_weights(w, "gated")
    for tile in each_tile(monkeypatch):
        assert torch.equal(o.gemm_float_gated(a, w, split=split), want), tile


@pytest.mark.parametrize("heads,kv_heads,d,bs", [(4, 2, 64, 16), (3, 1, 48, 32)])
def test_rotary_product_from_parts(heads, kv_heads, d, bs, monkeypatch):
    o = ops()
    m, k = 100, 512
    a, w = rnd(m, k, seed=5).cuda(), rnd((heads + 2 * kv_heads) * d, k, seed=6).cuda()
    slots = torch.randperm(2 * m, generator=torch.Generator().manual_seed(7))[:m].to(torch.int32).cuda()
    cos, sin = (rnd(m, d // 2, seed=s).cuda() for s in (8, 9))
    split = o.float_split_weights(w, "rotary", d)

    def product(split):
        k_pages, v_pages = torch.zeros((2 * m // bs + 1, kv_heads, bs, d), device="cuda"), torch.zeros((2 * m // bs + 1, kv_heads, d, bs), device="cuda")
        q = o.gemm_float_rotary(a, w, dict(positions=torch.arange(m, dtype=torch.int32, device="cuda"), cos=cos, sin=sin, slots=slots, k_pages=k_pages,
                                           v_pages=v_pages, num_heads=heads, num_kv_heads=kv_heads, head_dim=d, block_size=bs), split)
        return q, k_pages, v_pages
    want = product(None)
    for tile in each_tile(monkeypatch):
        assert all(torch.equal(x, y) for x, y in zip(product(split), want)), tile


def test_results_that_are_not_finite_from_parts(monkeypatch):
    """Infinities, NaN and numbers past the largest bfloat16 among rows and weights: made again from the floats, as without the parts."""
    o = ops()
    a, w = rnd(70, 1030, seed=10), rnd(50, 1030, seed=11)
    a[1, 3], w[2, 1029], w[3, 0], a[4] = float("inf"), float("-inf"), float("nan"), a[4] * 2.0 ** -120
    a[2, :], w[4, :] = 0.0, 0.0
    a[2, 5], w[4, 5] = 3.4e38, 0.5
    a, w = a.cuda(), w.cuda()
    a, w = a[:, :1028], w[:, :1028]                       # (rows with a stride of their own: not on 16-byte boundaries, and so from the floats)
    split = o.float_split_weights(w)
    for tile in each_tile(monkeypatch):
        assert o.gemm_float_split(a, w, split) is None
        x, y = a.contiguous(), w.contiguous()
        got, want = o.gemm_float_split(x, y, split), o.gemm_generic(x, y)
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(nan=0.0), want.nan_to_num(nan=0.0)), tile


# one row, rows and weight rows past the last tile, tiles of 16 x 16 and 16 x 32, a last slice of one column
@pytest.mark.parametrize("m,n,k", [(1, 16, 512), (8, 2048, 2048), (17, 1030, 1000), (24, 2048, 993), (16, 4090, 2044)])
def test_product_as_two_sums(m, n, k):
    o = ops()
    a, w = rnd(m, k, seed=12).cuda(), rnd(n, k, seed=13).cuda()
    a[0, 0], a[0, k - 1] = float("inf"), float("nan")
    halves, want = o.gemm_float_halves(a, w), o.gemm_generic(a, w)
    assert halves.shape == (2, m, n) and bool(want[0].isnan().all()) and bool(halves[1, 0].isnan().all()) and not bool(halves[0, 0].isfinite().any())
    assert torch.equal((halves[0] + halves[1])[1:], want[1:])
    a[0] = 1.0
    assert torch.equal(o.gemm_float_halves(a, w).sum(0)[:1], o.gemm_generic(a, w)[:1])


def test_which_products_come_as_two_sums():
    o = ops()
    assert o.float_halves_plan(8, 2048, 2048, 256) == 1 and o.float_halves_plan(24, 2048, 2048, 256) == o.float_halves_plan(8, 4096, 2048, 256) == 2
    assert o.float_halves_plan(33, 2048, 2048, 256) is None and o.float_halves_plan(8, 2048, 520, 256) is None       # (too many tiles; slices without columns)


def test_which_products_take_the_parts():
    o = ops()
    assert o.float_split_plan(95, 2048, 2048, 256) is None and o.float_split_plan(301, 2048, 480, 256) is None
    assert o.float_split_plan(301, 2048, 2048, 256) == (3, 4) and o.float_split_plan(301, 11264, 2048, 256) == (4, 4)
    assert o.float_split_plan(128, 2048, 2048, 256) is None               # (tiles of 32 x 32 from the floats are ahead)


@pytest.mark.parametrize("pairing,n", [("plain", 1 << 20), ("plain", (1 << 20) - 15), ("gated", 1 << 20)])
def test_parts_of_as_many_rows_as_a_matrix_may_have(pairing, n):
    """65,536 tiles of 16 rows, one more than a grid has: the last rows' parts are those of a matrix of these rows alone."""
    o = ops()
    w = torch.zeros(n, 32, device="cuda")
    last = rnd(40, 32, seed=14).cuda()
    w[-40:] = last
    assert o.float_split_takes(w)
    parts = o.float_split_weights(w, pairing)
    if pairing == "plain":
        few = o.float_split_weights(w[(n - 40) // 16 * 16:])
        assert parts.shape[0] == (n + 15) // 16 and torch.equal(parts[-few.shape[0]:].view(torch.int16), few.view(torch.int16))
    else:
        gate, up = torch.zeros(48, 32, device="cuda"), w[-48:]
        assert torch.equal(parts[-6:].view(torch.int16), o.float_split_weights(torch.cat([gate, up]), "gated").view(torch.int16))
    del parts, w
    torch.cuda.empty_cache()


def test_a_matrix_has_its_parts_from_the_first_product_on_that_is_faster_from_them(monkeypatch):
    """Not for few rows, short rows or another epilogue, not inside a capture, and not past the share of the memory; the product's bits are the same."""
    from paged_llm_amd.parts import linear as L
    o = ops()
    w, x = rnd(2048, 2048, seed=15).cuda(), rnd(301, 2048, seed=16).cuda()
    want = o.gemm_generic(x, w)
    matrix = L.Weight(w)
    assert torch.equal(L.linear(x[:8], matrix), o.gemm_generic(x[:8], w)) and matrix._parts is None
    assert matrix.parts(301, "gated") is None and L.Weight(w[:, :480].contiguous()).parts(301, "plain") is None
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=stream):
        captured = L.linear(x, matrix)
    graph.replay()
    assert torch.equal(captured, want) and matrix._parts is None
    with torch.cuda.stream(stream):
        made = L.linear(x, matrix)
    assert matrix._parts is not None and torch.equal(L.linear(x, matrix), want)          # (another stream than the one that made them)
    stream.synchronize()
    assert torch.equal(made, want)
    for share in (0.0, 0.25):
        monkeypatch.setattr(L.Weight, "PARTS_MEMORY_SHARE", share)
        other = L.Weight(w)
        assert torch.equal(L.linear(x, other), want) and (other._parts is None) == (share == 0.0)

    def out_of_memory(*a):
        raise torch.OutOfMemoryError
    monkeypatch.setattr(o, "float_split_weights", out_of_memory)
    other = L.Weight(w)
    assert torch.equal(L.linear(x, other), want) and other._parts is None and other.parts(301, "plain") is None


def test_several_threads_ask_for_the_parts_at_once():
    import threading

    from paged_llm_amd.parts import linear as L
    o = ops()
    w, x = rnd(2048, 2048, seed=17).cuda(), rnd(301, 2048, seed=18).cuda()
    want, matrix, got = o.gemm_generic(x, w), L.Weight(w), [None] * 6
    torch.cuda.synchronize()

    def product(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            got[i] = L.linear(x, matrix)
        stream.synchronize()
    threads = [threading.Thread(target=product, args=(i,)) for i in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(torch.equal(y, want) for y in got)


def test_what_a_model_lays_out_with_its_first_step_counts_once_for_the_cache_pool(monkeypatch):
    """A probing step that leaves 1 GB behind and needs 100 MB for itself: as many pages as when the 1 GB is there already."""
    from types import SimpleNamespace

    from paged_llm_amd.engine import pool_sizing
    from paged_llm_amd.engine.loading import random_model
    from tests.tiny_configs import TINY_A
    model = random_model(TINY_A, dtype="float32")
    left = []

    def probe(*args):
        torch.empty(100 << 20, dtype=torch.uint8, device="cuda")
        if not left:
            left.append(torch.empty(1 << 30, dtype=torch.uint8, device="cuda"))
    monkeypatch.setattr(pool_sizing, "_probe_step", probe)
    config = SimpleNamespace(block_size=16, max_num_batched_tokens=64, max_num_seqs=1 << 20, max_model_len=1 << 20, gpu_memory_utilization=0.9)
    page = sum(g.bytes_per_page(16, model.dtype) for g in model.cache_groups().values())
    pages = [pool_sizing.pages_that_fit(model, config) for _ in range(2)]
    assert abs(pages[0] - pages[1]) * page < 200 << 20
