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


def taken(runner, *lengths, **kind):
    """Portion tokens of the graph that the step is replayed from; None: eagerly."""
    entry = runner._prompt_graph(portions(*lengths, **kind))
    return None if entry is None else entry["key"][3]


def test_a_step_shares_a_graph_until_its_own_shape_has_paid_for_one():
    """140 tokens: in the shape of 192 from the second time on, in their own of 160 once 32 rows of padding were computed 50 times (as many as ten
    steps of 160 hold); 180 tokens fill their own shape and the shared one alike."""
    runner = runner_for()
    assert [taken(runner, 140) for _ in range(49)] == [None] + [192] * 48
    assert [taken(runner, 140) for _ in range(3)] == [160] * 3 and taken(runner, 180) == 192 and taken(runner, 192) == 192
    assert [k[3] for k in runner.captured] == [192, 160]


def test_graphs_beyond_a_thousand_tokens():
    """Where a shared shape is filled exactly, and own shapes that come back again and again: not those of wide models with linear recurrences, for
    which a padding sequence is a chunk more."""
    plain, narrow, wide = runner_for(width=2048), runner_for(width=1024), runner_for(width=1025)
    narrow.padding_is_a_chunk = wide.padding_is_a_chunk = True
    for runner in (plain, narrow):
        assert [taken(runner, 1100) for _ in range(101)] == [None] * 99 + [1104] * 2
    assert [taken(wide, 1100) for _ in range(200)] == [None] * 200 and [taken(wide, 1104) for _ in range(101)] == [None] * 99 + [1104] * 2
    for runner in (plain, narrow, wide):
        assert [taken(runner, 2048) for _ in range(3)] == [None, 2048, 2048] and [taken(runner, 1280) for _ in range(3)] == [None, 1280, 1280]
        assert [taken(runner, 2050) for _ in range(200)] == [None] * 200


def test_which_models_say_that_padding_is_a_chunk():
    from paged_llm_amd.engine.loading import build_model
    from tests.gudutar_configs import GUDU_A
    from tests.mekusun_configs import MEKU_A
    from tests.tiny_configs import TINY_A
    assert build_model(GUDU_A, "bfloat16", "cpu").padding_is_a_chunk()
    assert not build_model(MEKU_A, "bfloat16", "cpu").padding_is_a_chunk() and not build_model(TINY_A, "bfloat16", "cpu").padding_is_a_chunk()


def test_a_stream_of_prompts_of_every_length_captures_few_shapes():
    """500 prompts of 16 to 2,048 tokens: no more captures than there are shared shapes (14 up to 1,024 tokens, four filled exactly beyond), and most steps
    up to 1,024 tokens are replayed."""
    import random
    for width in (1024, 2048):
        rng, runner = random.Random(5), runner_for(width=width)
        lengths = [rng.randint(16, 2048) for _ in range(500)]
        replayed = sum(taken(runner, n) is not None for n in lengths)
        assert len(runner.captured) <= 18 and len(set(runner.captured)) == len(runner.captured)
        assert replayed >= sum(n <= 1024 for n in lengths) - 18
    scored = runner_for()
    for n in lengths:
        taken(scored, n, want="all")
    assert len(scored.captured) <= 18


def test_a_shape_that_had_to_go_waits_before_it_takes_anothers_place():
    runner = runner_for(per_kind=1)
    assert [taken(runner, 30) for _ in range(3)] == [None, 32, 32] and [taken(runner, 60) for _ in range(2)] == [None, 64]
    assert [taken(runner, 30) for _ in range(19)] == [None] * 17 + [32] * 2


def test_the_warm_up_of_a_shape_stays_within_its_bound():
    """Its portions are as long as one another, so none has positions that the model has no tables for: four portions of 26 tokens, all that a model
    of 26 positions takes, share a shape of 128 tokens with a padding sequence, of 26 each at most."""
    for positions in (17, 26, 39, 40, 64, 100, 256):
        runner = runner_for(max_positions=positions)
        for count in (1, 2, 3, 4):
            for n in range(2, positions + 1):
                for shared in (True, False):
                    key = runner._prompt_graph_key(portions(*[n] * count), shared=shared)
                    if key is not None:
                        each = runner._even_portions(key[3], count + 1)
                        assert sum(each) == key[3] and max(each) <= key[5] <= positions, (positions, count, n)
