"""Prompts whose tokens all want logits, replayed from graphs (the session captures a shape when it first sees it): more wanted rows than a graph holds logits
for, lengths that share a graph, and results that a later replay leaves alone."""

import pytest
import torch

from tests import helpers
from tests.helpers import TraceBuilder
from tests.test_replay_gpu import check, folders, session_for  # noqa: F401  (a fixture)
from tests.tiny_configs import TINY_A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_texts_scored_again_and_again(folders, dtype):  # noqa: F811
    folder = folders["A", dtype]
    lengths = [150, 150, 150, 131, 160, 64, 64, 64, 65, 65, 65, 150]
    reqs = {f"r{i}": helpers.random_tokens(n, TINY_A["vocab_size"], seed=40 + i) for i, n in enumerate(lengths)}
    session = session_for(folder, dtype, 192)
    trace = TraceBuilder()
    for rid, toks in reqs.items():
        trace.step([(rid, toks, "all")], end=[rid])
    check(helpers.replay_in_process(session, trace), folder, reqs, dtype)
    graphs = [session.runner._graphs.get(k) for k in list(session.runner._graphs) if k[0] == "prompt"]
    assert {"head_rows" in g for g in graphs} == {True, False}, "one shape wants 64 rows of logits or fewer, the others more"


def test_logits_of_a_replay_are_the_callers(folders):  # noqa: F811
    """Two steps through one graph: the first one's logits stay as they are, and come out the same when it runs again."""
    session = session_for(folders["A", "bfloat16"], "bfloat16", 192)
    runner, manager = session.runner, session.manager
    from paged_llm_amd.engine.batch import StepEntry

    def step(rid, tokens):
        assert manager.allocate(rid, 0, len(tokens))
        tables, slot, version = manager.step_fields(rid)
        out = runner.step([StepEntry(rid, tokens, 0, {g: list(t) for g, t in tables.items()}, slot, list(range(len(tokens))), version)])
        manager.free(rid)
        return out
    texts = [helpers.random_tokens(n, TINY_A["vocab_size"], seed=n) for n in (140, 155)]
    for i in range(3):
        step(f"w{i}", texts[0])
    first = step("a", texts[0])
    kept = first.clone()
    other = step("b", texts[1])
    assert first.shape == (140, TINY_A["vocab_size"]) and other.shape == (155, TINY_A["vocab_size"]) and torch.equal(first, kept)
    assert torch.equal(step("c", texts[0]), kept)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_portions_that_hold_more_tokens_than_the_context_bound(folders, dtype):  # noqa: F811
    """Four portions together longer than any position of the model, replayed from one graph and, between the replays, run eagerly: the same
    logits up to the type's rounding (a padded step's products may take other tiles)."""
    from paged_llm_amd.engine.batch import StepEntry
    from paged_llm_amd.engine.loading import build_runtime, load_model
    from tests.test_replay_gpu import TOL
    model = load_model(folders["A", dtype], dtype, "cuda")
    manager, _, runner = build_runtime(model, 16, 80, 8, enable_prefix_caching=False, use_graphs=True, graph_after_sightings=1)

    def logits(lengths, graphs):
        entries = []
        for i, n in enumerate(lengths):
            assert manager.allocate(i, 0, n)
            tables, slot, version = manager.step_fields(i)
            entries.append(StepEntry(i, helpers.random_tokens(n, TINY_A["vocab_size"], seed=n + i), 0, {g: list(t) for g, t in tables.items()}, slot,
                                     [0, n - 1], version))
        runner.prompt_graphs = True
        key = runner._prompt_graph_key(entries, shared=True)
        assert key[3] > key[5] == model.max_positions
        runner.prompt_graphs = graphs
        out = runner.step(entries)
        for i in range(len(lengths)):
            manager.free(i)
        return out
    for lengths in [(100, 101, 99, 90), (60, 130, 120, 111), (2, 200, 100, 96), (100, 101, 99, 90)]:
        got, want = logits(lengths, True), logits(lengths, False)
        assert (got - want).abs().max() <= TOL[dtype] * want.abs().max()
    assert [k[0] for k in runner._graphs] == ["prompt"], "one shape holds them all"


@pytest.mark.parametrize("tokens", [1, 40])
def test_a_capture_leaves_the_graphs_of_a_runner_that_is_gone_alone(folders, tokens):  # noqa: F811
    """A runner that only a cycle keeps, dropped while another one captures: its graphs go with a later collection."""
    import gc
    from paged_llm_amd.engine.batch import StepEntry
    from paged_llm_amd.engine.loading import build_runtime, load_model
    model = load_model(folders["A", "bfloat16"], "bfloat16", "cuda")

    def stepped(n):
        manager, _, runner = build_runtime(model, 16, 16, 2, enable_prefix_caching=False, use_graphs=True, graph_after_sightings=1)
        assert manager.allocate(0, 0, n)
        tables, slot, version = manager.step_fields(0)
        return runner, runner.step([StepEntry(0, [5] * n, 0, {g: list(t) for g, t in tables.items()}, slot, [n - 1], version)])
    gone, want = stepped(tokens)
    gone.itself = gone
    held, forward = [gone], model.forward
    del gone

    def dropping(*args, **kwargs):
        if torch.cuda.is_current_stream_capturing() and held:
            held.clear()
            [[i] for i in range(100000)]                    # (so many containers start a collection)
            assert not gc.isenabled()
        return forward(*args, **kwargs)
    model.forward = dropping
    try:
        runner, got = stepped(tokens)
    finally:
        del model.forward
    assert not held and len(runner._graphs) == 1 and gc.isenabled() and torch.equal(got, want)
