"""What a step of the slot scheduler takes (batching.py): tokens of every kind that torch's conversion takes, in eager steps and in replayed ones alike."""
import pytest
import torch

import revitar_oracle as O
from gbx_lm_amd.batching import BatchScheduler
from gbx_lm_amd.utils import load_model

DEVICES = ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)]
CONFIG = O.make_config([O.attention_layer(4, 2, 32, 32, window=16, mlp=O.moe(4, 2, 32))], vocab=50, width=64)


@pytest.fixture(scope="module")
def path(tmp_path_factory):
    return O.save_checkpoint(str(tmp_path_factory.mktemp("steps")), CONFIG, O.make_weights(CONFIG, 1))


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("form", ["device tensors", "host tensors", "floats", "numpy"])
def test_decode_steps_take_what_their_first_ones_take(path, device, form):
    """The third step of a set of slots is the first that a graph replays."""
    import numpy as np
    model = load_model(path, device=device, dtype=torch.float32)[0]
    made = {"device tensors": lambda t: torch.tensor(t, device=device), "host tensors": torch.tensor, "floats": float, "numpy": np.int32}[form]
    plain, other = BatchScheduler(model), BatchScheduler(model)
    for i in range(6):
        tokens = [(7 * i + j) % 50 for j in range(2)]
        a = plain.step([(j, [t]) for j, t in enumerate(tokens)])
        b = other.step([(j, [made(t)]) for j, t in enumerate(tokens)])
        assert torch.equal(a, b)


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("put", ["subclass", "object", "class"])
def test_generate_goes_through_a_step_put_in_its_place(path, device, put, monkeypatch):
    """A subclass's, an object's or the class's own replaced step sees every step, and its logits last as long as it keeps them."""
    model = load_model(path, device=device, dtype=torch.float32)[0]
    prompts, seen = [[3, 1, 4], [1, 5]], []
    want = BatchScheduler(model).generate(prompts, max_tokens=7)
    step = BatchScheduler.step

    def watched(self, entries, want=None):
        logits = step(self, entries, want)
        seen.append((logits, logits.clone()))
        return logits

    eng = type("Watched", (BatchScheduler,), {"step": watched})(model) if put == "subclass" else BatchScheduler(model)
    if put == "object":
        eng.step = lambda entries, want=None: watched(eng, entries, want)
    elif put == "class":
        monkeypatch.setattr(BatchScheduler, "step", watched)
    assert eng.generate(prompts, max_tokens=7) == want
    assert len(seen) == 7 and all(torch.equal(a, b) for a, b in seen)


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("pos0,n_new,q_tile,error", [([0], [2.0], 128, TypeError), ([0], [3], 0, ValueError), ([2 ** 31 - 2], [3], 128, RuntimeError)])
def test_tables_of_impossible_steps_are_refused(device, pos0, n_new, q_tile, error):
    """Rows that are no whole number, tiles without a row, positions past the tables' 32 bits."""
    from gbx_lm_amd.batching import StepBatch
    with pytest.raises(error):
        StepBatch.build([1], pos0, n_new, device, q_tile)
