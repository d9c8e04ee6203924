"""The tokens of a prompt step on the host: checked one by one or as an array, turned into an array once at the most."""
import types

import numpy as np
import pytest


@pytest.fixture
def engine(monkeypatch):
    """An engine's step function without a device: what fill is handed and how many arrays were made."""
    from bitnet_c_amd.engine import step
    made, filled = [], []
    monkeypatch.setattr(step, "np", types.SimpleNamespace(
        array=lambda x: made.append(len(x)) or np.array(x), concatenate=np.concatenate))
    graph = types.SimpleNamespace(fill=lambda slots, tokens, *rest: filled.append([int(t) for t in tokens]), upload=lambda: None,
                                  run=lambda: np.zeros((64, 1)).view(type("Logits", (np.ndarray,), {"clone": np.copy})))
    eng = object.__new__(step.Engine)
    eng.cache = types.SimpleNamespace(length=lambda slot: 0)
    eng.vocab_size, eng.max_seq_len = 389, 5000
    eng._prompt_graph_for = lambda key: graph

    def run(prompts):
        made.clear(), filled.clear()
        entries = [step.StepEntry(i, p, [len(p) - 1]) for i, p in enumerate(prompts)]
        arrays = eng._validate(entries)
        eng._step_prompt_graph(entries, arrays, list(range(len(prompts))), [len(p) for p in prompts], [0] * len(prompts))
        assert filled == [[int(t) for p in prompts for t in p]]
        return sorted(made)
    return run


def _prompt(n):
    return [(7 * i) % 389 for i in range(n)]


def test_a_prompt_becomes_an_array_once_and_a_short_one_never(engine):
    from bitnet_c_amd.engine.step import ARRAY_TOKENS as N
    assert engine([_prompt(2)] * 8) == [] and engine([_prompt(N - 1)]) == []
    assert engine([_prompt(N)]) == [N] and engine([_prompt(2000), _prompt(3), _prompt(N)]) == [N, 2000]


@pytest.mark.parametrize("odd", [tuple, np.array, lambda p: [np.int64(t) for t in p], lambda p: [bool(p[0])] + p[1:], lambda p: [float(t) for t in p],
                                 lambda p: [str(t) for t in p]])
def test_other_kinds_of_tokens_give_the_same_numbers(engine, odd):
    for n in (2, 200):
        engine([odd(_prompt(n)), _prompt(100), _prompt(2)])


@pytest.mark.parametrize("n", [3, 200])
@pytest.mark.parametrize("bad", [-1, 389, 2 ** 40, 2 ** 63, 2 ** 70, -2 ** 63, 400.5])
def test_a_token_outside_the_vocabulary_is_named(engine, n, bad):
    from bitnet_c_amd.engine import StepError
    for at in (0, n // 2, n - 1):
        p = _prompt(n)
        p[at] = bad
        with pytest.raises(StepError, match="slot 1: token .* is outside") as e:
            engine([_prompt(100), p])
        assert f"token {bad} " in str(e.value)
