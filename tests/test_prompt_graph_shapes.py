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


# ------------------------------------------------------------------------------ which graph a step takes, and when one is captured
def runner_for(max_positions=4096, width=None, per_kind=64):
    """A runner whose captures only note the shape (no GPU here)."""
    import dataclasses
    from types import SimpleNamespace

    from paged_llm_amd.engine.loading import build_model, build_runtime
    from paged_llm_amd.weights.random_init import fill_random
    from tests.tiny_configs import TINY_A
    model = build_model(TINY_A, "bfloat16", "cpu", max_model_len=max_positions)
    fill_random(model, seed=0)
    model.max_positions = max_positions
    if width:
        model.spec = dataclasses.replace(model.spec, hidden_size=width)
    runner = build_runtime(model, 16, 8, 4, enable_prefix_caching=False)[2]
    runner.use_graphs = runner.prompt_graphs = True
    runner._graphs = GraphCache(per_kind)
    runner.captured = []
    runner._new_prompt_graph = lambda key: dict(key=key, copied=SimpleNamespace(synchronize=lambda: None))

    def capture(entry):
        runner.captured.append(entry["key"])
        return runner._graphs.put(entry["key"], entry)
    runner._capture_prompt_graph = capture
    return runner


def portions(*lengths, singles=0, want="last"):
    from paged_llm_amd.engine.batch import StepEntry
    return ([StepEntry(f"s{i}", [1], 20, {}, None, [0]) for i in range(singles)]
            + [StepEntry(f"p{i}", [1] * n, 0, {}, None, list(range(n)) if want == "all" else [n - 1]) for i, n in enumerate(lengths)])


def test_the_warm_up_of_a_shape_stays_within_its_bound():
    """Its portions are as long as one another, so none has positions that the model has no tables for: four portions of 26 tokens, all that a model
    of 26 positions takes, share a shape of 128 tokens with a padding sequence, of 26 each at most."""
    for positions in (17, 26, 39, 40, 64, 100, 256):
        runner = runner_for(max_positions=positions)
        for count in (1, 2, 3, 4):
            for n in range(2, positions + 1):
                key = runner._prompt_graph_key(portions(*[n] * count))
                if key is not None:
                    each = runner._even_portions(key[3], count + 1)
                    assert sum(each) == key[3] and max(each) <= key[5] <= positions, (positions, count, n)
