"""The work whose speed matters to users of this package, as measurable cases.

Every case goes through the public entry points, as a program that uses the package calls them: ``generate()``, the
causal LM's forward (prompts with a kept state, scored text), a training step (loss and gradients of every parameter),
a single ``FusedBitLinear`` and the two scans with their gradients.  ``listed()`` names twelve of them, ``draw()`` makes
more of the same ranges.  Model shapes are the 370M (24 layers x 1024) and 1.3B (24 layers x 2048) rows of the model zoo.

``norms`` says what the norm weights hold.  "trained": every norm has weights of its own, as in any checkpoint that has
been trained (the three projections behind a block's norm then quantise three different rows).  "initial": all ones, as
a newly initialised model and the benchmark have them (the three projections share their quantised row).
"""
import math

import torch

import matmulfreellm_amd as mm

VOCAB = 32000
SHAPES = {"370M": (1024, 24), "1.3B": (2048, 24)}                 # hidden size, layers
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
TRAIN_LAYERS = 3                                                   # a training step returns every gradient: 50 tensors


# ------------------------------------------------------------------------------ the cases
def listed():
    return [
        # one row through one projection: the smallest call, nothing but latency
        {"name": "linear_1_row", "kind": "linear", "rows": 1, "k": 2048, "n": 2048, "dtype": "bf16"},
        # answering one user with a trained checkpoint, greedy
        {"name": "generate_1.3B_b1", "kind": "generate", "shape": "1.3B", "dtype": "bf16", "norms": "trained", "batch": 1,
         "prompt": 64, "new": 32, "sample": False},
        # the generation script's own options (half precision, top-p 0.4, temperature 0.6) for a handful of prompts of odd length
        {"name": "generate_370M_b5_sampled", "kind": "generate", "shape": "370M", "dtype": "fp16", "norms": "trained",
         "batch": 5, "prompt": 43, "new": 32, "sample": True},
        # serving many users at once; norm weights as the benchmark's batch-64 leg has them
        {"name": "generate_1.3B_b64", "kind": "generate", "shape": "1.3B", "dtype": "bf16", "norms": "initial", "batch": 64,
         "prompt": 32, "new": 32, "sample": False},
        # the time to the first token of a short prompt of odd length
        {"name": "prefill_370M_1x77", "kind": "prefill", "shape": "370M", "dtype": "bf16", "norms": "trained", "batch": 1,
         "tokens": 77, "padded": False},
        # a few prompts of different lengths, padded on the left
        {"name": "prefill_1.3B_3x459_padded", "kind": "prefill", "shape": "1.3B", "dtype": "fp16", "norms": "trained", "batch": 3,
         "tokens": 459, "padded": True},
        # long prompts in a batch, as the benchmark's prefill leg runs them: the largest call
        {"name": "prefill_1.3B_8x2048", "kind": "prefill", "shape": "1.3B", "dtype": "bf16", "norms": "initial", "batch": 8,
         "tokens": 2048, "padded": False},
        # scoring text (perplexity): logits of every position and their loss, no gradients
        {"name": "score_1.3B_2x1001", "kind": "score", "shape": "1.3B", "dtype": "bf16", "norms": "trained", "batch": 2,
         "tokens": 1001},
        # one training step of a large batch at the 1.3B width
        {"name": "train_2048_8x1024_bf16", "kind": "train", "hidden": 2048, "dtype": "bf16", "norms": "trained", "batch": 8,
         "tokens": 1024},
        # a small step in single precision, odd length (fine-tuning on short text)
        {"name": "train_1024_2x333_fp32", "kind": "train", "hidden": 1024, "dtype": "fp32", "norms": "trained", "batch": 2,
         "tokens": 333},
        # the scan of the reference's own timing table at its longest sequence, forward and backward
        {"name": "scan_chunk_16x4x16384x128", "kind": "scan", "op": "chunk", "batch": 16, "heads": 4, "tokens": 16384,
         "channels": 128, "dtype": "bf16", "state": False},
        # the recurrent form in single precision, carried state, odd sizes
        {"name": "scan_recurrent_3x5x777x96_fp32", "kind": "scan", "op": "recurrent", "batch": 3, "heads": 5, "tokens": 777,
         "channels": 96, "dtype": "fp32", "state": True},
    ]


def _log(rng, lo, hi):
    """A whole number, spread over its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["linear", "generate", "generate", "prefill", "prefill", "score", "train", "scan"])
    norms = rng.choice(["trained", "trained", "initial"])
    if kind == "linear":
        return {"kind": kind, "rows": _log(rng, 1, 8192), "k": 128 * _log(rng, 4, 44), "n": 32 * _log(rng, 16, 352),
                "dtype": rng.choice(["bf16", "fp16", "fp32"])}
    if kind == "generate":
        batch = _log(rng, 1, 64)
        return {"kind": kind, "shape": rng.choice(["370M", "1.3B"]), "dtype": rng.choice(["bf16", "bf16", "fp16"]), "norms": norms,
                "batch": batch, "prompt": _log(rng, 16, min(256, 4096 // batch)), "new": _log(rng, 16, 40),
                "sample": rng.random() < 0.4}
    if kind == "prefill":
        batch = _log(rng, 1, 16)
        return {"kind": kind, "shape": rng.choice(["370M", "1.3B"]), "dtype": rng.choice(["bf16", "bf16", "fp16"]), "norms": norms,
                "batch": batch, "tokens": _log(rng, 16, min(2048, 16384 // batch)), "padded": batch > 1 and rng.random() < 0.5}
    if kind == "score":
        batch = _log(rng, 1, 8)
        return {"kind": kind, "shape": rng.choice(["370M", "1.3B"]), "dtype": rng.choice(["bf16", "fp16"]), "norms": norms,
                "batch": batch, "tokens": _log(rng, 64, min(2048, 4096 // batch))}
    if kind == "train":
        batch = _log(rng, 1, 16)
        dtype = rng.choice(["bf16", "bf16", "fp32"])
        return {"kind": kind, "hidden": rng.choice([1024, 2048]), "dtype": dtype, "norms": norms, "batch": batch,
                "tokens": _log(rng, 128, min(2048, (8192 if dtype == "bf16" else 2048) // batch))}
    batch, heads, channels = _log(rng, 1, 16), _log(rng, 1, 8), 16 * _log(rng, 4, 128)
    most = max(64, min(16384, (1 << 27) // (batch * heads * channels)))
    return {"kind": "scan", "op": rng.choice(["chunk", "recurrent"]), "batch": batch, "heads": heads, "tokens": _log(rng, 64, most),
            "channels": channels, "dtype": rng.choice(["bf16", "bf16", "fp16", "fp32"]), "state": rng.random() < 0.4}


# ------------------------------------------------------------------------------ what a program has in hand
def _fill(model, norms, gen):
    """Weights N(0, 0.02) (the configuration's initializer_range); trained norm weights spread around one."""
    with torch.no_grad():
        for name, p in model.named_parameters():
            if name.endswith("lower_bounds"):
                p.copy_(torch.randn(p.shape, generator=gen, device=p.device))
            elif "norm" in name:
                p.fill_(1.0) if norms == "initial" else p.copy_(0.5 + torch.rand(p.shape, generator=gen, device=p.device))
            else:
                p.copy_(torch.randn(p.shape, generator=gen, device=p.device) * 0.02)


def _model(hidden, layers, dtype, norms, gen):
    with torch.device("meta"):
        model = mm.HGRNBitForCausalLM(mm.HGRNBitConfig(vocab_size=VOCAB, hidden_size=hidden, num_hidden_layers=layers))
    model = model.to(dtype).to_empty(device="cuda")
    _fill(model, norms, gen)
    return model


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind, dtype = case["kind"], DTYPES[case["dtype"]]
    state = {"case": case}
    if kind == "linear":
        layer = mm.FusedBitLinear(case["k"], case["n"]).to("cuda", dtype)
        _fill(layer, "trained", gen)
        layer.packed_weight()
        state["layer"] = layer
        state["x"] = torch.randn(case["rows"], case["k"], generator=gen, device="cuda").to(dtype)
    elif kind == "scan":
        shape = (case["batch"], case["heads"], case["tokens"], case["channels"])
        gate = torch.randn(shape, generator=gen, device="cuda") + 1.0
        gate = torch.nn.functional.logsigmoid(gate) if case["op"] == "chunk" else torch.sigmoid(gate)
        state["x"] = torch.randn(shape, generator=gen, device="cuda").to(dtype).requires_grad_()
        state["g"] = gate.to(dtype).requires_grad_()
        state["do"] = torch.randn(shape, generator=gen, device="cuda").to(dtype)
        state["h0"] = torch.randn(case["batch"], case["heads"], case["channels"], generator=gen, device="cuda") if case["state"] else None
    else:
        hidden, layers = SHAPES[case["shape"]] if "shape" in case else (case["hidden"], TRAIN_LAYERS)
        model = _model(hidden, layers, dtype, case["norms"], gen)
        tokens = case["prompt"] if kind == "generate" else case["tokens"]
        state["ids"] = torch.randint(0, VOCAB, (case["batch"], tokens), generator=gen, device="cuda")
        state["model"] = model.train() if kind == "train" else mm.pack_all(model.eval())
        if kind == "generate":
            state["sampler"] = torch.Generator(device="cuda").manual_seed(seed + 1)
        if case.get("padded"):
            pad = torch.randint(0, max(1, tokens // 2), (case["batch"], 1), generator=gen, device="cuda")
            state["mask"] = (torch.arange(tokens, device="cuda") >= pad).long()
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        with torch.no_grad():
            return state["layer"](state["x"])
    if kind == "generate":
        if case["sample"]:
            return state["model"].generate(state["ids"], max_new_tokens=case["new"], do_sample=True, top_p=0.4, temperature=0.6,
                                           generator=state["sampler"])
        return state["model"].generate(state["ids"], max_new_tokens=case["new"])
    if kind == "prefill":
        with torch.no_grad():
            out = state["model"](input_ids=state["ids"], attention_mask=state.get("mask"), use_cache=True, logits_to_keep=1)
        return [out.logits] + [layer[-1] for layer in out.past_key_values]
    if kind == "score":
        with torch.no_grad():
            out = state["model"](input_ids=state["ids"], labels=state["ids"], use_cache=False)
        return [out.loss, out.logits]
    if kind == "train":
        model = state["model"]
        model.zero_grad(set_to_none=True)
        loss = model(input_ids=state["ids"], labels=state["ids"]).loss
        loss.backward()
        return [loss.detach()] + [p.grad for p in model.parameters()]
    scan = mm.chunk_hgrn if case["op"] == "chunk" else mm.fused_recurrent_hgrn
    o, last = scan(state["x"], state["g"], initial_state=state["h0"], output_final_state=case["state"])
    dx, dg = torch.autograd.grad(o, (state["x"], state["g"]), state["do"])
    return [o.detach(), dx, dg] + ([last] if last is not None else [])


# ------------------------------------------------------------------------------ what a pass cannot do without
def _weights(hidden, layers):
    """Ternary weights of the blocks: i/f/g/o projections, gate/up, down."""
    inter = 256 * (-(-int(hidden * 8 / 3) // 256))
    return layers * (4 * hidden * hidden + 3 * hidden * inter)


def work(case):
    kind, e = case["kind"], DTYPES[case["dtype"]].itemsize
    if kind == "linear":
        m, k, n = case["rows"], case["k"], case["n"]
        return {"bytes": k * n / 4 + e * (m * k + m * n + k), "flops": 2 * m * k * n}
    if kind == "scan":
        # x, g, do in; o, dx, dg out
        count = case["batch"] * case["heads"] * case["tokens"] * case["channels"]
        return {"bytes": 6 * count * e, "flops": 6 * count}
    hidden, layers = SHAPES[case["shape"]] if "shape" in case else (case["hidden"], TRAIN_LAYERS)
    w, head, b = _weights(hidden, layers), hidden * VOCAB, case["batch"]
    state = 4 * b * layers * hidden                                # fp32 recurrent state
    if kind == "generate":
        # the prompt reads the 2-bit weights once, every further token once more, and the state in and out
        steps = case["new"] - 1
        return {"bytes": (steps + 1) * (w + head) / 4 + state * (1 + 2 * steps) + 8 * b * (case["prompt"] + case["new"]),
                "flops": 2 * b * ((case["prompt"] + steps) * w + (steps + 1) * head)}
    m = b * case["tokens"]
    if kind == "prefill":
        return {"bytes": (w + head) / 4 + m * (8 + hidden * e) + state + b * VOCAB * e, "flops": 2 * (m * w + b * head)}
    if kind == "score":
        return {"bytes": (w + head) / 4 + m * (16 + hidden * e) + m * VOCAB * e, "flops": 2 * m * (w + head)}
    # a training step reads the weights and writes their gradients; three contractions per weight
    return {"bytes": 2 * e * (w + 2 * head) + 16 * m, "flops": 6 * m * (w + head)}


def tolerance(case):
    kind, dtype = case["kind"], case["dtype"]
    if kind == "generate":
        return "exact"                                             # token ids
    if kind == "scan":
        return {"rel": 1e-5 if dtype == "fp32" else 1e-2}
    if kind == "train":
        # three layers of straight-through gradients, every tensor in between rounded to the parameters' type
        return {"rel": 1e-4 if dtype == "fp32" else 2e-2}
    return {"rel": 1e-5 if dtype == "fp32" else 1e-2}
