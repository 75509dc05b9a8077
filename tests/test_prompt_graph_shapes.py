"""Which prompt steps share a captured graph: the buckets of tokens and wanted rows, and what becomes of a graph that had to go."""

from paged_llm_amd.engine.runner import GraphCache, ModelRunner


def test_token_buckets():
    """Never below the tokens, never further above them than a step: 31 up to 1,024, 15 up to 2,048, 255 beyond."""
    for n in range(1, 6000):
        b = ModelRunner._token_bucket(n)
        assert 0 <= b - n <= (31 if n <= 1024 else 15 if n <= 2048 else 255) and ModelRunner._token_bucket(b) == b
    assert [ModelRunner._token_bucket(n) for n in (1, 32, 33, 777, 1025, 2049)] == [32, 32, 64, 800, 1040, 2304]


def test_the_cache_names_what_had_to_go():
    cache = GraphCache(per_kind=2)
    key = lambda n: ("prompt", 0, 1, n, 1, 512, 0)
    assert cache.put(key(32), "a") is None and cache.put(key(64), "b") is None and cache.put(key(64), "c") is None
    assert cache.get(key(32)) == "a" and cache.put(key(96), "d") == key(64) and key(64) not in cache and len(cache) == 2
