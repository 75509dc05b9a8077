"""Prompts whose tokens all want logits, replayed from graphs (from the third time a shape is seen): more wanted rows than a graph holds logits
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
