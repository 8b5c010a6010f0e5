"""A block's kernels launched by one call of the host against the same kernels called part by part: the same bits, in the logits and in
the pages, for every form that the products and the attention take, and refusals that leave the call to the parts."""

from __future__ import annotations

import pytest
import torch

from tokasaurus_amd.engine.batch import StepEntry
from tokasaurus_amd.engine.runner import ModelRunner
from tokasaurus_amd.kernels import ops
from tokasaurus_amd.parts import block

pytestmark = pytest.mark.gpu


def _config(width, heads, kv_heads, inner):
    return {"architectures": ["LlamaForCausalLM"], "model_type": "llama", "num_hidden_layers": 3, "hidden_size": width, "num_attention_heads": heads,
            "num_key_value_heads": kv_heads, "intermediate_size": inner, "vocab_size": 512, "rope_theta": 10000.0, "rms_norm_eps": 1e-5,
            "rope_scaling": None, "tie_word_embeddings": True, "max_position_embeddings": 8192}


CONFIGS = {"1b": _config(2048, 32, 8, 8192), "3b": _config(3072, 24, 8, 8192), "small": _config(1024, 16, 4, 1000)}

# of the steps below, the smallest whose blocks go in one call (fewer rows take products that no route of it names)
LEAST = {"1b": 17, "3b": 12, "small": 101}


def _steps(runner, prompts, rows, made=None):
    """Logits of a step of prompts beside decoding requests, and of a second portion of every prompt; what was ``made`` in front of them is
    forgotten."""
    gen = torch.Generator().manual_seed(1)
    draw = lambda n: torch.randint(0, 512, (n,), generator=gen).tolist()  # noqa: E731
    out = []
    for r in range(rows):
        runner.run([StepEntry(f"row-{r}", draw(40 + 300 * (r % 4)), [])])
    if made is not None:
        made.clear()
    for part in range(2):
        entries = [StepEntry(f"prompt-{i}", draw(n), [0, n - 1]) for i, n in enumerate(prompts)] + [StepEntry(f"row-{r}", draw(1), [0]) for r in range(rows)]
        out.append(runner.run(entries).logits.clone())
    return out


@pytest.mark.parametrize("name", list(CONFIGS))
@pytest.mark.parametrize("prompts,rows", [([12], 0), ([17], 0), ([40, 9], 0), ([64], 0), ([65], 3), ([101], 0), ([128, 1], 0), ([129], 0), ([256], 0),
                                          ([257], 2), ([300, 400], 0), ([1000], 20), ([1024], 0)])
def test_the_same_bits_as_part_by_part(name, prompts, rows, monkeypatch):
    made = []
    plan = block.BlockPlan.run
    monkeypatch.setattr(block.BlockPlan, "run", lambda self, *a: made.append(plan(self, *a)) or made[-1])
    results = []
    for most in (block.MOST_ROWS, 0):
        monkeypatch.setattr(block, "MOST_ROWS", most)
        runner = ModelRunner.from_random(CONFIGS[name], 3, "bfloat16", 16, 1200, 24, use_graphs=False)
        logits = _steps(runner, prompts, rows, made)
        results.append((logits, [t.clone() for group in (runner.storage.keys, runner.storage.values) for layers in group for t in layers]))
        # both steps, every layer but the last: its rows are those whose logits are wanted
        total = sum(prompts) + rows
        assert len(made) == (4 if LEAST[name] <= total <= most else 0) and all(m is not None for m in made)
        del runner
    torch.cuda.synchronize()
    for got, want in zip(*results):
        for g, w in zip(got, want):
            assert torch.equal(g, w)


@pytest.fixture
def made(monkeypatch):
    """What a block's call returned, call by call."""
    results, run = [], block.BlockPlan.run
    monkeypatch.setattr(block.BlockPlan, "run", lambda self, *a: results.append(run(self, *a)) or results[-1])
    return results


def _runner(change=lambda model: None, pages=400, requests=8):
    runner = ModelRunner.from_random(CONFIGS["1b"], 3, "bfloat16", 16, pages, requests, use_graphs=False)
    change(runner.model)
    return runner


def _other_positions(model):
    """The second layer's rotation by tables of its own, which turn the other way."""
    first = model.blocks[0].mixer.position
    other = model.blocks[1].mixer.position = type(first).__new__(type(first))
    other.__dict__.update(first.__dict__)
    other.sin = -first.sin


def _windows(model):
    for b, window in zip(model.blocks, (70, 0, 33)):
        b.mixer.window = window


@pytest.mark.parametrize("change,calls", [(_windows, 4), (_other_positions, 2)])
def test_layers_that_differ(change, calls, made, monkeypatch):
    """Windows of different sizes, each with a plan of its own; a layer with another position encoding goes part by part."""
    logits = []
    for most in (block.MOST_ROWS, 0):
        monkeypatch.setattr(block, "MOST_ROWS", most)
        logits.append(_steps(_runner(change), [100, 30], 3, made))
        assert len(made) == (calls if most else 0) and all(m is not None for m in made)
    plain = _steps(_runner(), [100, 30], 3)
    for got, want, other in zip(*logits, plain):
        assert torch.equal(got, want) and not torch.equal(got, other)


def test_on_another_stream_than_the_first(made):
    """Steps whose current stream is not the device's first: the kernels, and the memory between them, are that stream's."""
    want = _steps(_runner(), [100, 30], 3)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = _steps(_runner(), [100, 30], 3, made)
        assert len(made) == 4 and all(m is not None for m in made)
    side.synchronize()
    for g, w in zip(got, want):
        assert torch.equal(g, w)


def test_decoded_rows_cut_by_their_own_lengths():
    """Few long requests among short ones beside a prompt, whose keys are cut otherwise than where the same rows decode alone: other orders of
    32-bit sums in front of 8-bit roundings."""
    lengths = [300] * 10 + [4000] * 2
    assert ops.attention_even_split([n + 1 for n in lengths], 8, 64, 4) != ops.attention_split(4001, 12, 8, 64, 4)
    logits = []
    for prompt in ([], [StepEntry("prompt", list(range(40)), [])]):
        runner = _runner(pages=900, requests=16)
        gen = torch.Generator().manual_seed(2)
        draw = lambda n: torch.randint(0, 512, (n,), generator=gen).tolist()  # noqa: E731
        for r, n in enumerate(lengths):
            runner.run([StepEntry(f"row-{r}", draw(n), [])])
        logits.append(runner.run(prompt + [StepEntry(f"row-{r}", [7 * r], [0]) for r in range(len(lengths))]).logits.float().clone())
        del runner
    alone, beside = logits
    assert ((beside - alone).norm(dim=1) <= 0.02 * alone.norm(dim=1)).all()


def test_what_does_not_lie_as_the_kernels_read_it_goes_part_by_part(monkeypatch):
    """A norm's weight that starts 2 bytes behind a multiple of 16: the parts take it, in the same kernels but one."""
    made = []
    plan = block.BlockPlan.run
    monkeypatch.setattr(block.BlockPlan, "run", lambda self, *a: made.append(plan(self, *a)) or made[-1])
    runner = ModelRunner.from_random(CONFIGS["1b"], 3, "bfloat16", 16, 100, 4, use_graphs=False)
    want = _steps(runner, [100], 0)
    assert made and all(m is not None for m in made)
    runner.release("prompt-0")
    made.clear()
    norm = runner.model.blocks[0].ff_norm
    moved = torch.empty(2049, dtype=norm.weight.dtype, device="cuda")[1:]
    moved.copy_(norm.weight)
    norm.weight = moved
    got = _steps(runner, [100], 0)
    assert made[0] is None and made[1] is not None
    for g, w in zip(got, want):
        assert float((g - w).norm() / w.norm()) < 0.02  # (other kernels for one projection: the order of 32-bit sums in front of 8-bit roundings)


def test_a_steps_memory_goes_back_with_the_step():
    """The plan and its memory end with the step, with the collector off."""
    import gc

    runner = ModelRunner.from_random(CONFIGS["1b"], 3, "bfloat16", 16, 100, 4, use_graphs=False)
    runner.run([StepEntry("a", list(range(100)), [])])
    gc.collect()
    gc.disable()
    try:
        held = []
        for i in range(6):
            runner.release("a")
            runner.run([StepEntry("a", list(range(100)), [])])
            held.append(torch.cuda.memory_allocated())
    finally:
        gc.enable()
    assert held[-1] == held[1]
