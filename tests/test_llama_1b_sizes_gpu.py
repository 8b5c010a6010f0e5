"""The layer sizes of Llama-3.2-1B (hidden 2048, 32 heads over 8 kv heads of 64, intermediate
8192, a vocabulary of 128256, llama3 rotary scaling, tied head) with two layers and random
weights: the sizes the kernels are tuned for, against the plain implementation, in 32-bit and
in bfloat16, a long request with its last tokens one by one and mixed batches on few pages."""

import pytest
import torch

import plain_llama
from gpu_common import TOL
from replay_helpers import compare, faulty_tail, mixed_trace, run_steps, shift_position, swap_pages
from tiny_models import make_folder, random_tokens, sharpen
from tokasaurus_amd.engine.runner import ModelRunner

pytestmark = pytest.mark.gpu

CONFIG_1B_SIZES = {
    "architectures": ["LlamaForCausalLM"],
    "model_type": "llama",
    "num_hidden_layers": 2,
    "hidden_size": 2048,
    "num_attention_heads": 32,
    "num_key_value_heads": 8,
    "intermediate_size": 8192,
    "vocab_size": 128256,
    "rope_theta": 500000.0,
    "rope_scaling": {
        "rope_type": "llama3",
        "factor": 32.0,
        "low_freq_factor": 1.0,
        "high_freq_factor": 4.0,
        "original_max_position_embeddings": 8192,
    },
    "rms_norm_eps": 1e-5,
    "tie_word_embeddings": True,
    "max_position_embeddings": 131072,
}
PAGE = 16
LONG = 600
MIXED = [90, 47, 130, 33, 71]
# logits are compared at these places of the long request's first step, and at every later place
LONG_WANT = [0, 1, 15, 16, 100, 255, 256, 511, 567]


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    folder = make_folder(tmp_path_factory.mktemp("llama_1b_sizes"), CONFIG_1B_SIZES, seed=3)
    V = CONFIG_1B_SIZES["vocab_size"]
    requests = {"long": random_tokens(LONG, V, 900)}
    requests.update({f"m{i}": random_tokens(n, V, 910 + i) for i, n in enumerate(MIXED)})
    cfg, w = plain_llama.load_folder(folder)
    plain = {rid: plain_llama.forward_logits(cfg, w, toks) for rid, toks in requests.items()}
    del w
    # the plain model computing in bfloat16 as the reference does: what the rounding alone costs
    cfg, w16 = plain_llama.load_folder(folder, torch.bfloat16)
    plain16 = {rid: plain_llama.forward_logits(cfg, w16, toks) for rid, toks in requests.items()}
    return folder, requests, plain, plain16


def errors(got, plain, other=None):
    """Root mean square and largest difference from the plain 32-bit logits over the rows of
    ``got``, of ``got`` itself or of the same rows of ``other``."""
    sq, n, worst = 0.0, 0, 0.0
    for (rid, pos), row in got.items():
        d = ((other[rid][pos] if other is not None else row) - plain[rid][pos]).double()
        sq += float((d * d).sum())
        n += d.numel()
        worst = max(worst, float(d.abs().max()))
    return (sq / n) ** 0.5, worst


def check_against_plain_bfloat16(got, plain, plain16, largest_too=True):
    """Six million logits through 2048-wide sums: the largest of so many rounding errors lies
    beyond what the tiny models' bound allows for a few thousand.  The measure here is the plain
    model computing in bfloat16 like the reference: the engine, which rounds in fewer places,
    must not be further from the 32-bit logits than that, over all rows and row for row
    (``largest_too``: also in the largest single error, a statistic for many rows only: the
    largest of six million errors is one logit's, which the two computations round alike up to
    the order of a sum (measured: 0.1254 or 0.1257 for the engine, by the order in which one
    product adds its terms, against 0.1256, with the same root mean square to four digits), so
    it may be a twentieth larger; a wrong page or position makes it several times larger)."""
    rms, worst = errors(got, plain)
    rms16, worst16 = errors(got, plain, plain16)
    print(f"engine: rms error {rms:.3e}, largest {worst:.3e}; plain bfloat16: rms error {rms16:.3e}, largest {worst16:.3e}")
    assert rms <= rms16 and (worst <= 1.05 * worst16 or not largest_too), "further from the plain logits than the plain model in bfloat16"
    for key, row in got.items():
        r, _ = errors({key: row}, plain)
        r16, _ = errors({key: row}, plain, plain16)
        assert r <= 1.25 * r16, f"row {key}: {r:.3e} from the plain logits, the plain model in bfloat16 {r16:.3e}"


def long_steps(tokens):
    head = LONG - 32
    steps = [{"entries": [("long", tokens[:head], LONG_WANT)]}]
    steps += [{"entries": [("long", [t], [0])]} for t in tokens[head:]]
    steps[-1]["end"] = ["long"]
    return steps


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_long_request_and_mixed_batches(model, dtype):
    folder, requests, plain, plain16 = model
    # room for the long request, or for the four longest of the mixed ones: pages are used again
    runner = ModelRunner.from_folder(folder, dtype, page_size=PAGE, num_pages=-(-LONG // 64) * 64 // PAGE, max_slots=4)
    got = run_steps(runner, long_steps(requests["long"]))
    assert len(got) == len(LONG_WANT) + 32
    mixed = {rid: toks for rid, toks in requests.items() if rid != "long"}
    steps = mixed_trace(mixed, seed=5)
    assert max(len(s["entries"]) for s in steps) >= 3
    got.update(run_steps(runner, steps))
    assert len(got) == len(LONG_WANT) + 32 + sum(MIXED)
    if dtype == "float32":
        compare(got, plain, **TOL[dtype])
    else:
        check_against_plain_bfloat16(got, plain, plain16)
    assert runner.manager.num_free_pages() == [p.num_pages for p in runner.manager.pools]


@pytest.mark.parametrize("fault", ["none", "page", "position"])
def test_the_bfloat16_measure_finds_a_wrong_page_and_a_wrong_position(model, fault):
    """One page of 16 keys among 600 taken from another request, or a decoded token one
    position off: the measure that the bfloat16 run above passes must fail.  All reads stay
    inside pages the two requests own; without a fault the same steps pass."""
    folder, requests, plain, plain16 = model
    reqs = {"long": requests["long"], "m0": requests["m0"]}
    runner = ModelRunner.from_folder(folder, "bfloat16", page_size=PAGE, num_pages=(640 + 128) // PAGE, max_slots=4)
    faults = {"none": lambda r: None, "page": lambda r: swap_pages(r, "long", 7, "m0", 2),
              "position": lambda r: shift_position(r, "long")}
    got = faulty_tail(runner, reqs, "long", 8, faults[fault])
    if fault == "none":
        check_against_plain_bfloat16(got, plain, plain16, largest_too=False)
    else:
        with pytest.raises(AssertionError, match="plain"):
            check_against_plain_bfloat16(got, plain, plain16, largest_too=False)


def test_recorded_steps_of_many_rows_agree_with_eager_ones(model):
    """At these sizes a step takes other products than the tiny models' (split ones, gate and up streamed and in
    tiles, the library's for the head): every recorded size up to 128 rows, replayed with eager steps between, against an
    eager run."""
    from test_engine_gpu import recorded_against_eager

    folder = model[0]
    lengths = [3 + (5 * i) % 17 for i in range(136)]
    sizes = recorded_against_eager(folder, PAGE, CONFIG_1B_SIZES, 128, lengths, lambda i: 6 + (3 * i) % 23, budget=1024,
                                   padded=True)
    assert {32, 48, 64, 80, 96, 112, 128} <= sizes


def test_sixteen_layers_deep_in_bfloat16(tmp_path):
    """The depth of the 1B model (16 blocks, heads of 64 in groups of 4, llama3 scaling) at half its
    width: what sixteen blocks of bfloat16 rounding add up to.  Mixed batches on few pages and the
    last tokens one by one; every row must stay within twice the distance that the plain model
    computing in bfloat16 keeps from the plain 32-bit logits, and the 32-bit engine within the
    tiny models' bound."""
    from replay_helpers import compare_with_bfloat16_measure, tail_one_by_one

    cfg = dict(CONFIG_1B_SIZES, num_hidden_layers=16, hidden_size=1024, num_attention_heads=16, num_key_value_heads=4,
               intermediate_size=2816, vocab_size=3000, max_position_embeddings=4096)
    folder = make_folder(tmp_path / "deep", cfg, seed=8)
    requests = {f"d{i}": random_tokens(n, cfg["vocab_size"], 700 + i) for i, n in enumerate([150, 40, 97, 64])}
    pcfg, w = plain_llama.load_folder(folder)
    plain = {rid: plain_llama.forward_logits(pcfg, w, toks) for rid, toks in requests.items()}
    pcfg, w16 = plain_llama.load_folder(folder, torch.bfloat16)
    plain16 = {rid: plain_llama.forward_logits(pcfg, w16, toks) for rid, toks in requests.items()}
    for dtype in ("float32", "bfloat16"):
        runner = ModelRunner.from_folder(folder, dtype, page_size=PAGE, num_pages=(256 + 3 * 128) // PAGE, max_slots=4)
        got = run_steps(runner, mixed_trace(requests, seed=2))
        got.update(run_steps(runner, tail_one_by_one("d0", requests["d0"], 32)))
        assert len(got) == sum(len(t) for t in requests.values())
        if dtype == "float32":
            compare(got, plain, atol=2e-4, rtol=1e-3)  # sixteen blocks of 32-bit sums in another order
        else:
            worst = compare_with_bfloat16_measure(got, plain, plain16, **TOL[dtype])
            print(f"sixteen blocks in bfloat16: at most {worst:.2f} times the plain bfloat16 model's distance")
        assert runner.manager.num_free_pages() == [p.num_pages for p in runner.manager.pools]


def test_prompts_long_enough_for_each_form_of_the_prompt_attention(tmp_path, monkeypatch):
    """Which attention kernel a prompt portion takes depends on how many wavefronts it fills (at
    this shape one wavefront a token): paired tiles below 2 048, groups of tiles that share their
    loads with two sets of wavefronts from there, with one set from 3 072.  A prompt of 3 300
    tokens whole, its first 2 200 tokens whole, and the 3 300 in portions of 448 each take another
    one, at the engine's own thresholds, and the later portions have their keys cut into splits;
    rows across the prompt, at the portions' and the row tiles' edges and at its end, against the plain model (two layers, a small vocabulary: the head is not
    what is looked at).  Queries and keys are scaled so that few keys carry a row, values and the
    output projection so that the attention stands out of the residual stream: the plain model
    without the 300 farthest keys of the last rows must fail the same comparison."""
    from replay_helpers import compare_with_bfloat16_measure
    from tokasaurus_amd.kernels import ops

    cfg = dict(CONFIG_1B_SIZES, vocab_size=4096)
    folder = make_folder(tmp_path / "long_prompts", cfg, seed=8)
    sharpen(folder, {"v_proj.weight": 4.0, "o_proj.weight": 4.0})  # what the attention adds stands out of the residual stream
    tokens = random_tokens(3300, cfg["vocab_size"], 930)
    plain_cfg, w = plain_llama.load_folder(folder)
    plain = {"p": plain_llama.forward_logits(plain_cfg, w, tokens)}
    # the plain model without the 300 farthest keys of the last rows: what the comparison must tell from the right logits
    near = {"p": plain_llama.forward_logits(plain_cfg, w, tokens, windows={0: 3000, 1: 3000})}
    plain_cfg, w16 = plain_llama.load_folder(folder, torch.bfloat16)
    plain16 = {"p": plain_llama.forward_logits(plain_cfg, w16, tokens)}
    del w, w16

    forms: list = []
    real = ops.paged_attention_mfma

    def watching(*args, **kw):
        cut = args[14] < args[13]  # keys a split below the bound of the launch's requests
        forms.append("cut" if cut else int(kw.get("grouped", 0)))
        return real(*args, **kw)

    monkeypatch.setattr(ops, "paged_attention_mfma", watching)
    runner = ModelRunner.from_folder(folder, "bfloat16", page_size=PAGE, num_pages=2 * 3328 // PAGE, max_slots=2)
    want = [0, 1, 15, 16, 31, 32, 447, 448, 1000, 1023, 1024, 2047, 2048, 2198, 2199, 2200, 2687, 2688, 3135, 3136, 3298, 3299]

    def one_step(n):
        return [{"entries": [("p", tokens[:n], [p for p in want if p < n])], "end": ["p"]}]

    def in_portions(size):
        steps = [{"entries": [("p", tokens[at:at + size], [p - at for p in want if at <= p < at + size])]}
                 for at in range(0, len(tokens), size)]
        steps[-1]["end"] = ["p"]
        return steps

    # (the last portions of 448 tokens end after more than 2 048 keys: 448 wavefronts walking so far have their keys cut)
    for steps, form, rows in ((one_step(3300), {1}, len(want)), (one_step(2200), {2}, sum(p < 2200 for p in want)),
                              (in_portions(448), {0, "cut"}, len(want)), (in_portions(2200), {0, 2}, len(want))):
        forms.clear()
        got = run_steps(runner, steps)
        assert len(got) == rows and set(forms) == form, (form, set(forms))
        compare_with_bfloat16_measure(got, plain, plain16, **TOL["bfloat16"])
    # a short portion after a long past beside a whole prompt (the same tokens' first 700, so the same logits): planned
    # apart, the one with its keys cut, the other on paired tiles
    steps = in_portions(3236)[:1]
    steps.append({"entries": [("p", tokens[3236:], [p - 3236 for p in want if p >= 3236]), ("q", tokens[:700], [0, 31, 32, 447, 699])],
                  "end": ["p", "q"]})
    forms.clear()
    got = run_steps(runner, steps)
    assert {"cut", 0} <= set(forms), set(forms)
    both = lambda rows: {"p": rows["p"], "q": rows["p"]}
    compare_with_bfloat16_measure(got, both(plain), both(plain16), **TOL["bfloat16"])
    # two requests with the same tokens: both whole but for their ends in one step (grouped, one set), then a long and a
    # short portion after long pasts in one step: planned apart, the long one whole on paired tiles, the short one cut
    steps = [{"entries": [("p", tokens[:2700], [p for p in want if p < 2700]), ("q", tokens[:3236], [0, 2047, 3235])]},
             {"entries": [("p", tokens[2700:], [p - 2700 for p in want if p >= 2700]), ("q", tokens[3236:], [0, 63])], "end": ["p", "q"]}]
    forms.clear()
    got = run_steps(runner, steps)
    assert set(forms) == {1, 0, "cut"}, set(forms)
    compare_with_bfloat16_measure(got, both(plain), both(plain16), **TOL["bfloat16"])
    # logits as they would be with the far keys left out do not pass
    with pytest.raises(AssertionError, match="position 3299"):
        compare_with_bfloat16_measure({("p", 3299): near["p"][3299]}, plain, plain16, **TOL["bfloat16"])
