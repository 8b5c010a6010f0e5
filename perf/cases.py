"""Cases by which this engine's speed is measured: steps of the model runner and a whole generation.

A case is one model, one storage type and one kind of call:

``step``      one call of ``ModelRunner.run``: ``rows`` requests that hold ``context`` tokens each (with ``ragged``: from an
              eighth of it to all of it) decode one token, beside ``prompts`` new prompts of ``tokens`` tokens in all (ragged
              too when there are several).  rows alone: a decode step, replayed from a recording as the engine does it;
              prompts alone: a prefill; both: what a scheduler makes of requests that come while others decode.
``generate``  one call of ``Engine.generate``: ``prompts`` prompts of ``tokens`` tokens in all, ``new`` greedy tokens each, with
              the 20 most probable tokens of every step ranked.

Models have the layer sizes that ``bench.py`` names (Llama shapes of 1B, 3B and 8B whole; Kupuzen and Tefavik at the 1B
sizes with eight layers, as ``bench.py --design`` runs them) and random weights drawn from the seed.  Kupuzen stands for the
designs that keep a matrix a head instead of keys, Tefavik for those with mixtures of experts and two mixers side by side;
the designs whose routers choose experts by score are left out, since a rounding there changes whole rows.

Decoded tokens are given, not taken from the slot, and a bfloat16 step returns its logits alone though it samples: a near tie
that falls the other way is no error but would make the outputs incomparable.  Requests grow by a token a pass, as in use.
"""

import math

import torch

from tokasaurus_amd import EngineConfig, SamplingParams
from tokasaurus_amd.engine.batch import StepEntry
from tokasaurus_amd.engine.engine import Engine
from tokasaurus_amd.engine.runner import ModelRunner, Sampling
from tokasaurus_amd.models.registry import architecture_of, build_model

PAGE = 16
ROOM = 6144  # tokens a decoding request may grow by before its requests start again
RANKED = 20
DTYPES = {"bfloat16": torch.bfloat16, "float32": torch.float32}


# ---------------------------------------------------------------------------- models


def _llama(layers, width, heads, kv_heads, inner, factor, tied):
    return {"architectures": ["LlamaForCausalLM"], "model_type": "llama", "num_hidden_layers": layers, "hidden_size": width,
            "num_attention_heads": heads, "num_key_value_heads": kv_heads, "intermediate_size": inner, "vocab_size": 128256,
            "rope_theta": 500000.0, "rms_norm_eps": 1e-5, "tie_word_embeddings": tied, "max_position_embeddings": 131072,
            "rope_scaling": {"rope_type": "llama3", "factor": factor, "low_freq_factor": 1.0, "high_freq_factor": 4.0,
                             "original_max_position_embeddings": 8192}}


def _kupuzen():
    ff = {"kind": "dense", "ff": 8192}
    attention = {"type": "attention", "mlp": ff, "mixer": {
        "heads": 32, "kv_heads": 8, "dim": 64, "vdim": 64, "scale": 64 ** -0.5, "mask": {"size": 1024},
        "rot": {"base": 500000.0, "dims": 64, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}}}
    delta = {"type": "channel_delta", "mlp": ff, "mixer": {"heads": 16, "kv_heads": 16, "dim": 128, "vdim": 128, "conv": 4,
                                                           "decay_rank": 64, "gate_rank": 64}}
    return {"architecture": "Kupuzen", "vocab": 128256, "width": 2048, "embedding": {"scale": 1.0}, "norm": {"eps": 1e-6},
            "residual_mult": 1.0, "logit_softcap": 30.0, "layers": [attention if i % 4 == 3 else delta for i in range(8)]}


def _tefavik():
    mixture = {"kind": "moe", "expert": {"ff": 1024, "limit": 7.0}, "router": {"experts": 32, "top": 8}}
    gla = {"type": "gla", "mlp": mixture, "mixer": {"heads": 16, "dim": 128, "vdim": 128, "tau": 16.0, "rank": 16}}
    pair = {"type": "parallel", "mlp": mixture, "mixer": {
        "left": {"heads": 32, "kv_heads": 8, "dim": 64, "vdim": 64, "scale": 64 ** -0.5, "softcap": 50.0,
                 "mask": {"size": 1024}, "rot": {"base": 500000.0, "dims": 64}},
        "right": {"heads": 8, "dim": 128, "vdim": 128, "gate_cap": 15.0}}}
    return {"architecture": "Tefavik", "vocab": 128256, "width": 2048, "norm": {"eps": 1e-6},
            "loop": {"start": 1, "stop": 3, "times": 2}, "layers": [gla if i % 3 == 0 else pair for i in range(6)]}


MODELS = {"llama-1b": _llama(16, 2048, 32, 8, 8192, 32.0, True), "llama-3b": _llama(28, 3072, 24, 8, 8192, 32.0, True),
          "llama-8b": _llama(32, 4096, 32, 8, 14336, 8.0, False), "kupuzen-1b": _kupuzen(), "tefavik-1b": _tefavik()}


def _llama_shapes(c):
    W, inner, V = c["hidden_size"], c["intermediate_size"], c["vocab_size"]
    d = W // c["num_attention_heads"]
    kv = c["num_key_value_heads"] * d
    out = {"model.embed_tokens.weight": ((V, W), "matrix"), "model.norm.weight": ((W,), "signs")}
    if not c["tie_word_embeddings"]:
        out["lm_head.weight"] = ((V, W), "matrix")
    for i in range(c["num_hidden_layers"]):
        p = f"model.layers.{i}."
        for name, rows, cols in (("self_attn.q_proj", W, W), ("self_attn.k_proj", kv, W), ("self_attn.v_proj", kv, W),
                                 ("mlp.gate_proj", inner, W), ("mlp.up_proj", inner, W)):
            out[f"{p}{name}.weight"] = ((rows, cols), "matrix")
        out[f"{p}self_attn.o_proj.weight"], out[f"{p}mlp.down_proj.weight"] = ((W, W), 0.003), ((W, inner), 0.0025 / c["num_hidden_layers"])
        out[f"{p}input_layernorm.weight"] = out[f"{p}post_attention_layernorm.weight"] = ((W,), "norm")
    return out


def _kupuzen_shapes(c):
    W, V = c["width"], c["vocab"]
    out = {"embed": ((V, W), "matrix"), "head": ((V, W), "matrix"), "final.norm": ((W,), "offset")}
    for i, layer in enumerate(c["layers"]):
        m, p, ff = layer["mixer"], f"l{i}.mix.", layer["mlp"]["ff"]
        qk, kk, vv, H = m["heads"] * m["dim"], m["kv_heads"] * m["dim"], m["heads"] * m["vdim"], m["heads"]
        out[f"l{i}.norm1"] = out[f"l{i}.norm2"] = ((W,), "offset")
        out[f"l{i}.mlp.gate"] = out[f"l{i}.mlp.up"] = ((ff, W), "matrix")
        out[f"l{i}.mlp.down"] = ((W, ff), "matrix")
        out[p + "o"] = ((W, vv), "matrix")
        if layer["type"] == "attention":
            out.update({p + "q": ((qk, W), "matrix"), p + "k": ((kk, W), "matrix"), p + "v": ((m["kv_heads"] * m["vdim"], W), "matrix"),
                        p + "q.norm": ((qk,), "norm"), p + "k.norm": ((kk,), "norm"), p + "sink": ((H,), "vector")})
        else:
            r, g = m["decay_rank"], m["gate_rank"]
            out.update({p + "q": ((kk, W), "matrix"), p + "k": ((kk, W), "matrix"), p + "v": ((vv, W), "matrix"), p + "b": ((H, W), "matrix"),
                        p + "q.conv": ((kk, m["conv"]), "vector"), p + "k.conv": ((kk, m["conv"]), "vector"),
                        p + "v.conv": ((vv, m["conv"]), "vector"), p + "a1": ((r, W), "matrix"), p + "a2": ((qk, r), "matrix"),
                        p + "g1": ((g, W), "matrix"), p + "g2": ((vv, g), "matrix"), p + "A_log": ((H,), "vector"),
                        p + "dt_bias": ((qk,), "vector"), p + "norm": ((m["vdim"],), "norm")})
    return out


def _tefavik_shapes(c):
    W, V = c["width"], c["vocab"]
    out = {"embed": ((V, W), 1.0), "final.norm": ((W,), "small signs")}
    for i, layer in enumerate(c["layers"]):
        m, p, mlp = layer["mixer"], f"l{i}.mix.", layer["mlp"]
        out[f"l{i}.norm1"] = out[f"l{i}.norm2"] = ((W,), "norm")
        out[f"l{i}.mlp.table"] = ((V, mlp["router"]["top"]), mlp["router"]["experts"])
        for e in range(mlp["router"]["experts"]):
            out[f"l{i}.mlp.e{e}.gate"] = out[f"l{i}.mlp.e{e}.up"] = ((mlp["expert"]["ff"], W), "matrix")
            out[f"l{i}.mlp.e{e}.down"] = ((W, mlp["expert"]["ff"]), "matrix")
        if layer["type"] == "gla":
            qk, vv = m["heads"] * m["dim"], m["heads"] * m["vdim"]
            out.update({p + "q": ((qk, W), "matrix"), p + "k": ((qk, W), "matrix"), p + "v": ((vv, W), "matrix"), p + "g": ((vv, W), "matrix"),
                        p + "a1": ((m["rank"], W), "matrix"), p + "a2": ((qk, m["rank"]), "matrix"), p + "a2.b": ((qk,), "matrix"),
                        p + "norm": ((m["vdim"],), "norm"), p + "o": ((W, vv), "matrix")})
            continue
        a, b, pl, pr = m["left"], m["right"], p + "left.", p + "right."
        for name, rows in (("q", a["heads"] * a["dim"]), ("k", a["kv_heads"] * a["dim"]), ("v", a["kv_heads"] * a["vdim"])):
            out[pl + name], out[f"{pl}{name}.b"] = ((rows, W), "matrix"), ((rows,), "matrix")
        out.update({pl + "q.norm": ((a["dim"],), "norm"), pl + "k.norm": ((a["dim"],), "norm"), pl + "o": ((W, a["heads"] * a["vdim"]), "matrix"),
                    pl + "out": ((W,), "norm"), pr + "out": ((W,), "norm")})
        qk, vv = b["heads"] * b["dim"], b["heads"] * b["vdim"]
        out.update({pr + "q": ((qk, W), "matrix"), pr + "k": ((qk, W), "matrix"), pr + "v": ((vv, W), "matrix"), pr + "g": ((vv, W), "matrix"),
                    pr + "i": ((b["heads"], W), "matrix"), pr + "f": ((b["heads"], W), "matrix"), pr + "i.b": ((b["heads"],), "vector"),
                    pr + "f.b": ((b["heads"],), "vector"), pr + "norm": ((vv,), "norm"), pr + "o": ((W, vv), "matrix")})
    return out


SHAPES = {"llama": _llama_shapes, "kupuzen": _kupuzen_shapes, "tefavik": _tefavik_shapes}


def _family(case):
    return case["model"].split("-")[0]


def _vocab(case):
    c = MODELS[case["model"]]
    return c.get("vocab_size") or c["vocab"]


def _weights(case, seed):
    """Checkpoint tensors in bfloat16 on the GPU: matrices and their biases N(0, 0.02), norms 1 + N(0, 0.01) (N(0, 0.01) where
    they are stored around zero), other vectors N(0, 0.5), a table of experts' numbers that differ within a row.  A Llama's
    matrices that write into its 16-bit stream are smaller, so that no layer outweighs the embedding and every layer adds about
    as much: with 0.02 throughout, thirty layers turn the stream's roundings into 7 % of the logits, which no trained model
    does.  Tefavik's embedding is as large as what its normed mixers add, for the same reason.  Final norms in front of a tied
    head have random signs, so that it does not merely repeat the last token."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    out = {}
    for name, (shape, kind) in SHAPES[_family(case)](MODELS[case["model"]]).items():
        if isinstance(kind, int):
            keys = torch.rand((shape[0], kind), generator=gen, device="cuda")
            out[name] = keys.argsort(dim=-1)[:, : shape[1]].to(torch.int32).contiguous()
            continue
        t = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)
        t *= kind if isinstance(kind, float) else {"matrix": 0.02, "vector": 0.5}.get(kind, 0.01)
        if kind == "norm":
            t += 1.0
        elif kind in ("signs", "small signs"):
            t += torch.randint(0, 2, shape, generator=gen, device="cuda") * 2.0 - 1.0
            t *= 0.02 if kind == "small signs" else 1.0
        out[name] = t.to(torch.bfloat16)
    return out


# ---------------------------------------------------------------------------- the cases


def listed():
    def step(name, model, rows=0, context=0, prompts=0, tokens=0, ragged=False, dtype="bfloat16"):
        return {"name": name, "kind": "step", "model": model, "dtype": dtype, "rows": rows, "context": context, "prompts": prompts,
                "tokens": tokens, "ragged": ragged}

    return [
        step("1b_decode_1", "llama-1b", rows=1, context=1100),  # one user's chat: latency of a token
        step("1b_decode_8", "llama-1b", rows=8, context=6000),  # a few users with long contexts (the benchmark's batch)
        step("1b_decode_64_ragged", "llama-1b", rows=64, context=3000, ragged=True),  # a busy server, requests of all ages
        step("1b_prefill_2048", "llama-1b", prompts=1, tokens=2048),  # the benchmark's prompt
        step("1b_prefill_101", "llama-1b", prompts=1, tokens=101),  # a short question: time to the first token
        step("3b_mixed", "llama-3b", rows=45, context=2000, prompts=1, tokens=1000, ragged=True),  # a prompt arrives while others decode
        step("8b_decode_16_ragged", "llama-8b", rows=16, context=1500, ragged=True),  # the larger model, decoding
        step("8b_prefill_4x1024", "llama-8b", prompts=4, tokens=4096),  # prompts of several users in one step
        # a run in 32-bit, whole: scoring and checking against other implementations
        {"name": "1b_float32_generate", "kind": "generate", "model": "llama-1b", "dtype": "float32", "prompts": 4, "tokens": 301, "new": 8},
        step("kupuzen_prefill_1500", "kupuzen-1b", prompts=2, tokens=1500),  # recurrent layers over prompts
        step("kupuzen_decode_8", "kupuzen-1b", rows=8, context=2500),  # recurrent layers, one token a request
        step("tefavik_prefill_2048", "tefavik-1b", prompts=1, tokens=2048),  # experts and linear attention over a prompt
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["decode", "prefill", "mixed", "generate"], [0.4, 0.35, 0.15, 0.1])[0]
    if kind == "generate":
        prompts = rng.randint(1, 4)
        return {"kind": "generate", "model": "llama-1b", "dtype": "float32", "prompts": prompts, "tokens": _log_int(rng, 16 * prompts, 600),
                "new": rng.randint(3, 12)}
    model = rng.choices(list(MODELS), [0.4, 0.15, 0.15, 0.15, 0.15])[0]
    dtype = "float32" if model == "llama-1b" and rng.random() < 0.2 else "bfloat16"
    case = {"kind": "step", "model": model, "dtype": dtype, "rows": 0, "context": 0, "prompts": 0, "tokens": 0, "ragged": False}
    if kind != "prefill":
        held = {"llama-1b": 131072, "llama-8b": 24576}.get(model, 49152) // (4 if dtype == "float32" else 1)
        case["rows"] = _log_int(rng, 1, 64)
        case["context"] = _log_int(rng, 64, min(8192, held // case["rows"]))
        case["ragged"] = case["rows"] > 1 and rng.random() < 0.5
    if kind != "decode":
        most = {"llama-1b": 8192, "llama-3b": 4096, "llama-8b": 4000}.get(model, 3000) if kind == "prefill" else 1500
        case["tokens"] = _log_int(rng, 17, 600 if dtype == "float32" else most)
        case["prompts"] = rng.randint(1, min(6, case["tokens"] // 16))
    return case


def _spread(total, parts):
    """`parts` lengths that sum to `total`, the last about three times the first."""
    marks = [i * (1 + i / parts) / 2 for i in range(parts + 1)]
    cuts = [round(total * m / marks[-1]) for m in marks]
    return [b - a for a, b in zip(cuts, cuts[1:])]


def _held(case):
    """Tokens that every decoding request holds."""
    n, c = case.get("rows", 0), case.get("context", 0)
    return [max(1, c * (n + 7 * i) // (8 * n)) if case["ragged"] else c for i in range(1, n + 1)]


def _token_lists(case, seed, lengths):
    gen = torch.Generator().manual_seed(int(seed) * 2 + 1)
    return [torch.randint(0, _vocab(case), (n,), generator=gen).tolist() for n in lengths]


def _inputs(case, seed):
    """(what each decoding request holds, its next token beside the one that prepare() decodes, the prompts)."""
    held, prompts = _held(case) if case["kind"] == "step" else [], _spread(case["tokens"], case["prompts"]) if case["prompts"] else []
    got = _token_lists(case, seed, [n + 1 for n in held] + prompts)
    past = got[: len(held)]
    return [p[:-1] for p in past], [p[-1] for p in past], got[len(held):]


# ---------------------------------------------------------------------------- preparation and one pass


def prepare(case, seed):
    config = MODELS[case["model"]]
    arch = architecture_of(config)
    model = build_model(arch, arch.config_from_dict(config))
    weights = _weights(case, seed)
    model.load(weights, DTYPES[case["dtype"]], torch.device("cuda", torch.cuda.current_device()))
    del weights
    torch.cuda.empty_cache()
    past, following, prompts = _inputs(case, seed)
    if case["kind"] == "generate":
        longest = max(len(p) for p in prompts) + case["new"]
        pages = len(prompts) * -(-longest // PAGE)
        runner = ModelRunner(model, PAGE, pages, len(prompts), max_tokens_per_request=longest, topk_logprobs=RANKED)
        engine = Engine(EngineConfig(dtype=case["dtype"], page_size=PAGE, kv_cache_num_tokens=pages * PAGE, max_tokens_per_forward=1024,
                                     max_seqs_per_forward=len(prompts), max_topk_logprobs=RANKED, warmup_at_startup=False,
                                     stats_report_seconds=0, log_level="WARNING"), runner=runner)
        params = SamplingParams(temperature=0.0, max_tokens=case["new"], ignore_eos=True, topk_logprobs=RANKED)
        return {"kind": "generate", "engine": engine, "prompts": prompts, "params": params}
    room = max([len(p) + ROOM for p in past] + [0])
    longest = max([room] + [len(p) for p in prompts])
    pages = sum(-(-(len(p) + ROOM) // PAGE) for p in past) + sum(-(-len(p) // PAGE) for p in prompts)
    runner = ModelRunner(model, PAGE, pages, len(past) + len(prompts), max_tokens_per_request=longest)
    state = {"kind": "step", "runner": runner, "past": past, "room": [len(p) + ROOM for p in past], "dtype": case["dtype"],
             "portions": [StepEntry(f"prompt-{i}", p, [len(p) - 1]) for i, p in enumerate(prompts)],
             "decode": [StepEntry(f"row-{i}", [t], [0]) for i, t in enumerate(following)]}
    _fill(state)
    if past and not prompts:  # the step's recording is made at its first use
        runner.run(state["decode"], _greedy(len(past)))
    return state


def _greedy(n):
    return Sampling([0.0] * n, [0.0] * n)


def _fill(state):
    """The decoding requests' contexts, prefilled under a budget of tokens a step as the engine does it."""
    budget = 8192
    for i, tokens in enumerate(state["past"]):
        for at in range(0, len(tokens), budget):
            state["runner"].run([StepEntry(f"row-{i}", tokens[at:at + budget], [])])
    state["grown"] = 1


def run(state):
    if state["kind"] == "generate":
        done = state["engine"].generate(state["prompts"], state["params"])
        return {"tokens": torch.tensor([c.tokens for c in done]), "logprobs": torch.tensor([c.logprobs for c in done]),
                "ranked": torch.tensor([c.topk_ids for c in done]), "ranked_logprobs": torch.tensor([c.topk_logprobs for c in done])}
    runner = state["runner"]
    if state["grown"] + 1 >= ROOM:  # the requests have reached their length: others take their places
        for e in state["decode"]:
            runner.release(e.request_id)
        _fill(state)
    out = runner.run(state["portions"] + state["decode"], _greedy(len(state["portions"]) + len(state["decode"])))
    state["grown"] += 1
    for e in state["portions"]:  # a prompt's request ends, the next pass brings others
        runner.release(e.request_id)
    return {"logits": out.logits, "logprobs": out.logprobs, "ids": out.ids} if state["dtype"] == "float32" else {"logits": out.logits}


# ---------------------------------------------------------------------------- what a pass cannot do without


def _seen(n, window=0, section=0):
    """Keys that a query sees whose request holds n tokens with its own."""
    return (n - 1) % section + 1 if section else (min(n, window) if window else n)


def _run_order(config):
    n, loop = len(config["layers"]), config.get("loop")
    if not loop:
        return [(i, False) for i in range(n)]
    a, b, times = loop["start"], loop["stop"], loop["times"]
    return [(i, False) for i in range(a)] + [(i, t > 0 and i == a) for t in range(times) for i in range(a, b)] + [(i, False) for i in range(b, n)]


def _layers(case):
    """Per layer run: (layer, query heads, kv heads, head size, window, section, numbers of recurrent state)."""
    c = MODELS[case["model"]]
    if _family(case) == "llama":
        d = c["hidden_size"] // c["num_attention_heads"]
        return [(i, c["num_attention_heads"], c["num_key_value_heads"], d, 0, 0, 0) for i in range(c["num_hidden_layers"])]
    out = []
    for i, _ in _run_order(c):
        m, kind = c["layers"][i]["mixer"], c["layers"][i]["type"]
        if kind == "attention":
            out.append((i, m["heads"], m["kv_heads"], m["dim"], m["mask"]["size"], 0, 0))
        elif kind == "parallel":
            a, b = m["left"], m["right"]
            out.append((i, a["heads"], a["kv_heads"], a["dim"], 0, a["mask"]["size"], b["heads"] * b["dim"] * b["vdim"]))
        else:
            out.append((i, 0, 0, 0, 0, 0, m["heads"] * m["dim"] * m["vdim"]))
    return out


def work(case):
    size = 4 if case["dtype"] == "float32" else 2
    prompts = _spread(case["tokens"], case["prompts"]) if case["prompts"] else []
    if case["kind"] == "generate":
        steps = [([], prompts)] + [([n + j for n in prompts], []) for j in range(1, case["new"])]
    else:
        steps = [(_held(case), prompts)]
    shapes = SHAPES[_family(case)](MODELS[case["model"]])
    config = MODELS[case["model"]]
    V, W = _vocab(case), config.get("hidden_size") or config["width"]
    total = {"bytes": 0.0, "flops": 0.0}
    for rows, portions in steps:
        tokens, wants = len(rows) + sum(portions), len(rows) + len(portions)
        total["bytes"] += (V * W + tokens * W) * size + wants * V * 4
        total["flops"] += 2.0 * wants * V * W
        for i, heads, kv_heads, d, window, section, state in _layers(case):
            prefix = f"model.layers.{i}." if _family(case) == "llama" else f"l{i}."
            for name, (shape, kind) in shapes.items():
                if not name.startswith(prefix) or len(shape) < 2 or isinstance(kind, int):
                    continue
                share = config["layers"][i]["mlp"]["router"] if ".mlp.e" in name else None
                used = 1.0 if share is None else 1.0 - (1.0 - share["top"] / share["experts"]) ** tokens
                done = 1.0 if share is None else share["top"] / share["experts"]
                total["bytes"] += used * shape[0] * shape[1] * size
                total["flops"] += 2.0 * done * shape[0] * shape[1] * tokens
            pairs = sum(_seen(n + 1, window, section) for n in rows)
            kept = pairs + sum(portions)
            for n in portions:
                pairs += sum(_seen(j, window, section) for j in range(1, n + 1)) if window or section else n * (n + 1) // 2
            total["bytes"] += 2.0 * kept * kv_heads * d * size + 2.0 * (len(rows) + len(portions)) * state * 4
            total["flops"] += 4.0 * pairs * heads * d + 6.0 * tokens * state
    return total


def tolerance(case):
    # measured: with every product summed in another order (other kernels) the logits of a bfloat16 step move by 0.003 to
    # 0.016 of their norm and by up to 0.19 of their root mean square, and are 0.004 to 0.02 from the 64-bit ones; in 32-bit
    # they are 2e-6 to 3e-5 from them
    if case["dtype"] == "float32":
        return {"rel": 1e-4, "max": 4e-3, "differ": 0.01}
    return {"rel": 0.03, "max": 0.3}


# ---------------------------------------------------------------------------- the same in 64 bits, from the equations


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _product(x, w):
    """x w^T in 64 bits, many rows in pieces."""
    w = w.double().T
    return x @ w if x.shape[0] <= 32768 else torch.cat([part @ w for part in x.split(32768)])


def _frequencies(dims, base, scaling=None):
    f = base ** (-torch.arange(0, dims, 2, dtype=torch.float64, device="cuda") / dims)
    if scaling is None:
        return f
    factor, low, high, original = scaling
    turns = original * f / (2 * math.pi)
    t = (turns - low) / (high - low)
    return torch.where(turns < low, f / factor, torch.where(turns > high, f, (1 - t) * f / factor + t * f))


def _turn(x, positions, f, halves):
    """x [T, heads, d]; pair m is (m, m + d/2) with `halves`, else (2m, 2m + 1)."""
    a = positions.double()[:, None, None] * f
    c, s = torch.cos(a), torch.sin(a)
    u, v = x.chunk(2, -1) if halves else (x[..., 0::2], x[..., 1::2])
    pair = (u * c - v * s, v * c + u * s)
    return torch.cat(pair, -1) if halves else torch.stack(pair, -1).flatten(-2)


def _attend(q, k, v, scale, spans, window=0, section=0, softcap=0.0, sink=None):
    """q [T, H, d], k and v [T, G, d] of requests one after the other at `spans`."""
    out = torch.empty_like(q)
    each = q.shape[1] // k.shape[1]
    for a, b in spans:
        kk, vv = (t[a:b].repeat_interleave(each, 1).transpose(0, 1) for t in (k, v))
        at = torch.arange(b - a, device=q.device)
        for r in range(0, b - a, 1024):
            e = min(r + 1024, b - a)
            s = q[a + r:a + e].transpose(0, 1) @ kk[:, :e].transpose(1, 2) * scale
            if softcap:
                s = softcap * torch.tanh(s / softcap)
            i, j = at[r:e, None], at[None, :e]
            hidden = j > i
            if window:
                hidden = hidden | (i - j >= window)
            if section:
                hidden = hidden | (i // section != j // section)
            s = s.masked_fill(hidden, -math.inf)
            if sink is not None:
                s = torch.cat([s, sink[:, None, None].expand(-1, e - r, 1)], -1)
            p = torch.softmax(s, -1)[..., :e]
            out[a + r:a + e] = (p @ vv[:, :e]).transpose(0, 1)
    return out


def _padded(x, spans):
    """[T, ...] of requests one after the other -> [requests, longest, ...], zeros behind each."""
    out = x.new_zeros((len(spans), max(b - a for a, b in spans), *x.shape[1:]))
    for r, (a, b) in enumerate(spans):
        out[r, : b - a] = x[a:b]
    return out


def _flat(x, spans):
    return torch.cat([x[r, : b - a] for r, (a, b) in enumerate(spans)])


def _llama_stream(tokens, spans, w, c):
    H, G, eps = c["num_attention_heads"], c["num_key_value_heads"], c["rms_norm_eps"]
    d = c["hidden_size"] // H
    sc = c["rope_scaling"]
    f = _frequencies(d, c["rope_theta"], (sc["factor"], sc["low_freq_factor"], sc["high_freq_factor"], sc["original_max_position_embeddings"]))
    at = torch.cat([torch.arange(b - a, device="cuda") for a, b in spans])
    x = w["model.embed_tokens.weight"][tokens].double()
    for i in range(c["num_hidden_layers"]):
        p = f"model.layers.{i}."
        h = _rms(x, eps) * w[p + "input_layernorm.weight"].double()
        q, k, v = (_product(h, w[f"{p}self_attn.{n}_proj.weight"]).view(len(at), -1, d) for n in "qkv")
        o = _attend(_turn(q, at, f, True), _turn(k, at, f, True), v, d ** -0.5, spans)
        x = x + _product(o.flatten(1), w[p + "self_attn.o_proj.weight"])
        h = _rms(x, eps) * w[p + "post_attention_layernorm.weight"].double()
        x = x + torch.cat([_product(_silu(_product(part, w[p + "mlp.gate_proj.weight"])) * _product(part, w[p + "mlp.up_proj.weight"]),
                                    w[p + "mlp.down_proj.weight"]) for part in h.split(16384)])
    return _rms(x, eps) * w["model.norm.weight"].double(), w["model.embed_tokens.weight" if c["tie_word_embeddings"] else "lm_head.weight"]


def _delta(h, w, p, m, eps, spans):
    H, dk, dv, taps = m["heads"], m["dim"], m["vdim"], m["conv"]

    def conv(name):
        x = _padded(_product(h, w[p + name]), spans)
        taps_w = w[f"{p}{name}.conv"].double()
        x = torch.cat([x.new_zeros((x.shape[0], taps - 1, x.shape[2])), x], 1)
        n = x.shape[1] - taps + 1
        return _silu(sum(x[:, j:j + n] * taps_w[:, j] for j in range(taps))).unflatten(-1, (H, -1))

    unit = lambda x: x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    q, k, v = unit(conv("q")) * dk ** -0.5, unit(conv("k")), conv("v")
    beta = torch.sigmoid(_padded(_product(h, w[p + "b"]), spans))
    pre = _product(_product(h, w[p + "a1"]), w[p + "a2"]) + w[p + "dt_bias"].double()
    rate = torch.exp(w[p + "A_log"].double())[:, None]
    decay = _padded(torch.exp(-rate * torch.nn.functional.softplus(pre).unflatten(-1, (H, dk))), spans)
    S = h.new_zeros((len(spans), H, dk, dv))
    o = torch.empty_like(v)
    for t in range(v.shape[1]):
        S *= decay[:, t, :, :, None]
        u = beta[:, t, :, None] * (v[:, t] - (k[:, t, :, None, :] @ S)[..., 0, :])
        S += k[:, t, :, :, None] * u[..., None, :]
        o[:, t] = (q[:, t, :, None, :] @ S)[..., 0, :]
    gate = torch.sigmoid(_product(_product(h, w[p + "g1"]), w[p + "g2"])).unflatten(-1, (H, dv))
    return _product((_rms(_flat(o, spans), eps) * w[p + "norm"].double() * gate).flatten(1), w[p + "o"])


def _kupuzen_stream(tokens, spans, w, c):
    eps = c["norm"]["eps"]
    at = torch.cat([torch.arange(b - a, device="cuda") for a, b in spans])
    norm = lambda x, name: _rms(x, eps) * (1.0 + w[name].double())  # noqa: E731
    x = w["embed"][tokens].double()
    for i, layer in enumerate(c["layers"]):
        m, p = layer["mixer"], f"l{i}.mix."
        h = norm(x, f"l{i}.norm1")
        if layer["type"] == "attention":
            sc = m["rot"]["scaling"]
            f = _frequencies(m["dim"], m["rot"]["base"], (sc["factor"], sc["low"], sc["high"], sc["original"]))
            q, k = (_turn((_rms(_product(h, w[p + n]), eps) * w[f"{p}{n}.norm"].double()).view(len(at), -1, m["dim"]), at, f, False) for n in "qk")
            v = _product(h, w[p + "v"]).view(len(at), -1, m["vdim"])
            o = _attend(q, k, v, m["scale"], spans, window=m["mask"]["size"], sink=w[p + "sink"].double())
            y = _product(o.flatten(1), w[p + "o"])
        else:
            y = _delta(h, w, p, m, eps, spans)
        h = norm(x, f"l{i}.norm2")
        x = x + y + _product(_silu(_product(h, w[f"l{i}.mlp.gate"])) * _product(h, w[f"l{i}.mlp.up"]), w[f"l{i}.mlp.down"])
    return norm(x, "final.norm"), w["head"]


def _gated_linear(h, w, p, m, eps, spans):
    H, d, dv = m["heads"], m["dim"], m["vdim"]
    q, k, v = (_padded(_product(h, w[p + n]).unflatten(-1, (H, -1)), spans) for n in "qkv")
    q = q * d ** -0.5
    z = _product(_product(h, w[p + "a1"]), w[p + "a2"]) + w[p + "a2.b"].double()
    a = _padded(torch.exp(torch.nn.functional.logsigmoid(z) / m["tau"]).unflatten(-1, (H, d)), spans)
    S = h.new_zeros((len(spans), H, d, dv))
    o = torch.empty_like(v)
    for t in range(v.shape[1]):
        S = a[:, t, :, :, None] * S + k[:, t, :, :, None] * v[:, t, :, None, :]
        o[:, t] = (q[:, t, :, None, :] @ S)[..., 0, :]
    o = (_rms(_flat(o, spans), eps) * w[p + "norm"].double()).flatten(1)
    return _product(o * _silu(_product(h, w[p + "g"])), w[p + "o"])


def _matrix_memory(h, w, p, m, eps, spans):
    H, d, cap = m["heads"], m["dim"], m["gate_cap"]
    q, k, v = (_padded(_product(h, w[p + n]).unflatten(-1, (H, -1)), spans) for n in "qkv")
    q = q * d ** -0.5
    i, f = (_padded(cap * torch.tanh((_product(h, w[p + n]) + w[f"{p}{n}.b"].double()) / cap), spans) for n in "if")
    f = torch.nn.functional.logsigmoid(f)
    S, n = h.new_zeros((len(spans), H, d, m["vdim"])), h.new_zeros((len(spans), H, d))
    top = h.new_zeros((len(spans), H))
    o = torch.empty_like(v)
    for t in range(v.shape[1]):
        new = torch.maximum(f[:, t] + top, i[:, t])
        keep, write = torch.exp(f[:, t] + top - new)[..., None], torch.exp(i[:, t] - new)[..., None]
        S = keep[..., None] * S + (write * k[:, t])[..., None] * v[:, t, :, None, :]
        n = keep * n + write * k[:, t]
        top = new
        below = torch.maximum((n * q[:, t]).sum(-1).abs(), torch.exp(-top)) + 1e-6
        o[:, t] = (q[:, t, :, None, :] @ S)[..., 0, :] / below[..., None]
    o = _rms(_flat(o, spans), eps).flatten(1) * w[p + "norm"].double()
    return _product(o * torch.sigmoid(_product(h, w[p + "g"])), w[p + "o"])


def _tefavik_stream(tokens, spans, w, c):
    eps = c["norm"]["eps"]
    at = torch.cat([torch.arange(b - a, device="cuda") for a, b in spans])
    norm = lambda x, name: _rms(x, eps) * w[name].double()  # noqa: E731
    x0 = x = w["embed"][tokens].double()
    for i, add in _run_order(c):
        layer, p, q_ = c["layers"][i], f"l{i}.mix.", f"l{i}.mlp."
        m = layer["mixer"]
        x = x + x0 if add else x
        h = norm(x, f"l{i}.norm1")
        if layer["type"] == "gla":
            x = x + _gated_linear(h, w, p, m, eps, spans)
        else:
            a, pl = m["left"], p + "left."
            q, k, v = ((_product(h, w[pl + n]) + w[f"{pl}{n}.b"].double()).unflatten(-1, (-1, a["dim"])) for n in "qkv")
            f = _frequencies(a["dim"], a["rot"]["base"])
            q, k = (_turn(norm(t, f"{pl}{n}.norm"), at, f, False) for t, n in ((q, "q"), (k, "k")))
            o = _attend(q, k, v, a["scale"], spans, section=a["mask"]["size"], softcap=a["softcap"], sink=q.new_zeros(a["heads"]))
            left = norm(_product(o.flatten(1), w[pl + "o"]), pl + "out")
            right = norm(_matrix_memory(h, w, p + "right.", m["right"], eps, spans), p + "right.out")
            x = x + 0.5 * (left + right)
        h = norm(x, f"l{i}.norm2")
        chosen, limit = w[q_ + "table"][tokens], layer["mlp"]["expert"]["limit"]
        for e in range(layer["mlp"]["router"]["experts"]):
            rows = (chosen == e).any(-1).nonzero()[:, 0]
            g = torch.clamp(_product(h[rows], w[f"{q_}e{e}.gate"]), max=limit)
            u = torch.clamp(_product(h[rows], w[f"{q_}e{e}.up"]), -limit, limit)
            y = _product(g * torch.sigmoid(1.702 * g) * (u + 1), w[f"{q_}e{e}.down"])
            x = x.index_add(0, rows, y / layer["mlp"]["router"]["top"])
    return norm(x, "final.norm"), w["embed"]


STREAMS = {"llama": _llama_stream, "kupuzen": _kupuzen_stream, "tefavik": _tefavik_stream}


def _last_logits(case, w, sequences):
    """Logits behind the last token of every sequence."""
    ends = torch.tensor([len(s) for s in sequences]).cumsum(0).tolist()
    spans = [(e - len(s), e) for s, e in zip(sequences, ends)]
    tokens = torch.tensor([t for s in sequences for t in s], device="cuda")
    config = MODELS[case["model"]]
    h, head = STREAMS[_family(case)](tokens, spans, w, config)
    logits = _product(h[[e - 1 for e in ends]], head)
    cap = config.get("logit_softcap")
    return cap * torch.tanh(logits / cap) if cap else logits


def exact(case, seed):
    past, following, prompts = _inputs(case, seed)
    params = sum(s[0] * s[1] for s, kind in SHAPES[_family(case)](MODELS[case["model"]]).values() if len(s) == 2 and not isinstance(kind, int))
    if 2.0 * params * (sum(map(len, past)) + sum(map(len, prompts))) > 4.5e14:  # more than some twenty seconds in 64 bits
        return None
    w = _weights(case, seed)
    if case["kind"] == "generate":
        sequences, tokens, rows = [list(p) for p in prompts], [], []
        for _ in range(case["new"]):
            rows.append(torch.log_softmax(_last_logits(case, w, sequences), -1))
            tokens.append(rows[-1].argmax(-1))
            for s, t in zip(sequences, tokens[-1].tolist()):
                s.append(t)
        lp, chosen = torch.stack(rows, 1), torch.stack(tokens, 1)
        top = lp.topk(RANKED, -1)
        return {"tokens": chosen, "logprobs": lp.gather(-1, chosen[..., None])[..., 0], "ranked": top.indices, "ranked_logprobs": top.values}
    # (a step of decoded tokens alone has been run once before: its recording was made then)
    twice = [1] if prompts else [1, 1]
    logits = _last_logits(case, w, prompts + [p + [t] * len(twice) for p, t in zip(past, following)])
    if case["dtype"] == "bfloat16":
        return {"logits": logits}
    lp = torch.log_softmax(logits, -1)
    return {"logits": logits, "logprobs": lp.max(-1).values, "ids": lp.argmax(-1)}
