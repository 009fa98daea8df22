"""Timed workloads of this framework: what its users have it do, through its public entry points.

A case is a dict of plain values.  ``listed()`` names the fixed ones, ``draw(rng)`` gives one
more of the same ranges, ``prepare(case, seed)`` makes what a program holds before the call,
``run(state)`` is one pass, ``work(case)`` counts what a pass cannot do without and
``tolerance(case)`` says how far another correct implementation may be off.

Five kinds of work are covered:

* ``train``: hard forward and surrogate backward of ``rosa_soft`` / ``rosa_soft_varlen``, the
  gradient of the output coming from the layers above;
* ``forward``: the same operators without gradients (evaluation, frozen layers);
* ``prefill``: a prompt handed to a fresh ``RosaRuntime`` in one update;
* ``generate``: a prompt and then decoding updates of one or a few tokens per slot;
* ``project``: the hard forward in bit form and the output projection that reads the bits.
"""

from __future__ import annotations

import math

import torch

import rosa_soft_amd
from rosa_soft_amd import cabi

DEVICE = "cuda:0"
ITEM_BYTES = {"float32": 4, "float16": 2, "bfloat16": 2}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def _operator(kind, name, dtype, H, D, Hv, Dv, W, p=0.0, ms=3.0, B=0, T=0, lengths="",
              pattern="random"):
    case = dict(kind=kind, dtype=dtype, B=B, T=T, lengths=lengths, H=H, D=D, Hv=Hv, Dv=Dv, W=W,
                pattern=pattern)
    if kind == "train":
        case.update(p=p, ms=ms)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # the smallest model that is trained in earnest: a step is a handful of launches
        _operator("train", "train_tiny", "float32", H=4, D=4, Hv=4, Dv=8, W=16, B=1, T=256),
        # a short-context training step with grouped value heads and dropout
        _operator("train", "train_grouped", "float32", H=64, D=8, Hv=16, Dv=8, W=128, p=0.1,
                  B=2, T=1024),
        # the training step that the headline throughput is quoted on
        _operator("train", "train_metric", "float32", H=64, D=8, Hv=16, Dv=8, W=128, p=0.1,
                  B=2, T=4096),
        # mixed-precision training with wide values, one value head per query head
        _operator("train", "train_wide", "bfloat16", H=32, D=16, Hv=32, Dv=64, W=32, B=4, T=4096),
        # repetitive text: few symbols, matches as long as the window, one long sequence
        _operator("train", "train_long_match", "float16", H=16, D=2, Hv=16, Dv=32, W=256,
                  B=1, T=8192, pattern="motif"),
        # a packed batch of long documents in mixed precision; the largest step
        _operator("train", "train_packed", "bfloat16", H=64, D=32, Hv=8, Dv=32, W=64, p=0.1,
                  ms=9.0, lengths="1024,7168,2048,4096,512,8192,3072,6656"),
        # a packed batch of samples as they come: odd lengths, one of a single token, odd widths
        _operator("train", "train_ragged", "float32", H=12, D=12, Hv=6, Dv=24, W=48, p=0.1,
                  lengths="1,37,129,513,1000,2047,3001"),
        # evaluation at the shape of the headline training step
        _operator("forward", "forward_metric", "float32", H=64, D=8, Hv=16, Dv=8, W=128,
                  B=2, T=4096),
        # one short evaluation sample with odd sizes: nothing but latency
        _operator("forward", "forward_odd", "float16", H=9, D=5, Hv=3, Dv=20, W=33, B=1, T=333),
        # serving: two prompts of 4096 tokens arrive as logits, the routed values leave as such
        dict(name="prefill", kind="prefill", dtype="bfloat16", logits=True, S=2, T=4096, H=64,
             Hp=16, qk_bits=8, payload_bits=8, W=128, pattern="random"),
        # serving: eight slots with prompts of 4096 tokens, then 64 tokens one by one
        dict(name="generate", kind="generate", dtype="float32", logits=False, S=8, T=4096, H=64,
             Hp=16, qk_bits=8, payload_bits=8, W=128, steps=64, chunk=1, pattern="random"),
        # the operator and the projection behind it, without the expanded activation between them
        dict(name="project", kind="project", dtype="bfloat16", B=4, T=4096, H=32, D=16, Hv=32,
             Dv=64, W=32, N=2048),
    ]


def _spread(rng, low, high):
    """An integer between the bounds, even over the logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


MOST_PAIRS = 2_000_000_000  # (row, route) pairs of a drawn training step
MOST_ROWS = 2_000_000       # tokens x heads of any drawn case


def draw(rng):
    kind = rng.choice(["train"] * 5 + ["forward"] * 2 + ["prefill", "generate", "project"])
    if kind in ("train", "forward"):
        value_heads = _spread(rng, 1, 32)
        heads = value_heads * rng.choice([1, 1, 2, 4])
        # a context of some length, as many of them as the limits leave room for
        longest = _spread(rng, 64, 8192)
        pairs = MOST_PAIRS if kind == "train" else 4 * MOST_PAIRS
        room = min(MOST_ROWS // (heads * longest), pairs * 2 // (heads * longest * longest), 16)
        count = _spread(rng, 1, max(1, room))
        case = _operator(
            kind, "", rng.choice(["float32", "float16", "bfloat16"]), H=heads,
            D=rng.choice([2, 4, 5, 7, 8, 8, 12, 16, 16, 24, 32]), Hv=value_heads,
            Dv=rng.choice([8, 8, 12, 16, 20, 32, 32, 33, 48, 64]), W=_spread(rng, 8, 256),
            p=rng.choice([0.0, 0.1, 0.2]), ms=rng.choice([3.0, 9.0]),
            pattern=rng.choice(["random", "random", "motif"]))
        if rng.random() < 0.4:
            case["lengths"] = ",".join(
                str(longest if i == 0 else _spread(rng, 1, longest)) for i in range(count))
        else:
            case.update(B=count, T=longest)
        return case
    if kind in ("prefill", "generate"):
        payload_heads = _spread(rng, 1, 16)
        heads = payload_heads * rng.choice([1, 2, 4])
        tokens = _spread(rng, 64, 8192)
        case = dict(kind=kind, dtype=rng.choice(["float32", "bfloat16"]),
                    logits=rng.random() < 0.5,
                    S=_spread(rng, 1, max(1, min(16, MOST_ROWS // (tokens * heads)))),
                    T=tokens, H=heads, Hp=payload_heads, qk_bits=rng.choice([4, 6, 8, 8]),
                    payload_bits=rng.choice([4, 8, 8]), W=_spread(rng, 16, 256),
                    pattern=rng.choice(["random", "motif"]))
        if kind == "generate":
            case.update(steps=_spread(rng, 8, 64), chunk=rng.choice([1, 1, 1, 2, 4]))
        return case
    value_heads = rng.choice([4, 8, 16, 32])
    return dict(kind=kind, dtype="bfloat16", B=rng.randint(1, 4), T=_spread(rng, 128, 4096),
                H=value_heads * rng.choice([1, 2]), D=rng.choice([8, 12, 16]), Hv=value_heads,
                Dv=rng.choice([8, 16, 32, 64] if value_heads < 32 else [8, 16, 32]),
                W=_spread(rng, 16, 128), N=64 * _spread(rng, 8, 40))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _lengths(case):
    if case.get("lengths"):
        return [int(item) for item in case["lengths"].split(",")]
    return [case["T"]] * case["B"]


def _logits(generator, shape, dtype, pattern):
    """Query and key logits of ``[..., T, H, bits]``: independent, or (``motif``) keys that
    repeat a motif of 64 tokens with a tenth of the positions flipped, and queries close to
    them, as repetitive text gives."""

    randn = lambda *dims: torch.randn(*dims, device=DEVICE, generator=generator)
    if pattern == "random":
        return randn(*shape).to(dtype), randn(*shape).to(dtype)
    *batch, tokens, heads, bits = shape
    motif = randn(*batch, 64, heads, bits)
    repeats = [1] * len(batch) + [-(-tokens // 64), 1, 1]
    key = motif.repeat(*repeats)[..., :tokens, :, :]
    flip = torch.rand(*batch, tokens, heads, 1, device=DEVICE, generator=generator) < 0.10
    key = torch.where(flip, -key, key).to(dtype)
    return (key.float() + 0.1 * randn(*shape)).to(dtype), key


def _symbols(logits, bits):
    weights = 2 ** torch.arange(bits, device=DEVICE)
    return ((logits > 0) * weights).sum(-1).to(torch.uint8)


def prepare(case, seed):
    generator = torch.Generator(device=DEVICE).manual_seed(int(seed))
    dtype = getattr(torch, case["dtype"])
    randn = lambda *dims: torch.randn(*dims, device=DEVICE, generator=generator).to(dtype)
    kind = case["kind"]
    if kind in ("train", "forward"):
        lengths = _lengths(case)
        lead = (sum(lengths),) if case["lengths"] else (case["B"], case["T"])
        query, key = _logits(generator, (*lead, case["H"], case["D"]), dtype, case["pattern"])
        value = randn(*lead, case["Hv"], case["Dv"])
        arguments, offsets = [query, key, value], None
        if case["lengths"]:
            ends = torch.tensor([0, *lengths], dtype=torch.int32).cumsum(0, dtype=torch.int32)
            offsets = ends.to(DEVICE)
        controls = dict(max_suffix_length=case["W"])
        state = dict(kind=kind, arguments=arguments, offsets=offsets, controls=controls)
        if kind == "train":
            controls.update(scale=1.0, dropout_p=case["p"], mismatch_scale=case["ms"])
            for leaf in arguments:
                leaf.requires_grad_()
            # the gradient that the layers above hand to the operator's output
            state.update(grad_output=randn(*lead, case["H"], case["Dv"]), seed=int(seed))
        return state
    if kind == "project":
        shape = (case["B"], case["T"])
        depth = case["H"] * case["Dv"]
        weight = torch.randn(case["N"], depth, device=DEVICE, generator=generator) / depth ** 0.5
        return dict(
            kind=kind, controls=case["W"], value_dim=case["Dv"], weight=weight.to(dtype),
            arguments=[randn(*shape, case["H"], case["D"]), randn(*shape, case["H"], case["D"]),
                       randn(*shape, case["Hv"], case["Dv"])],
            residual=randn(*shape, case["N"]))
    # a runtime and the streams of its slots: the prompt, then the decoding chunks
    steps, chunk = case.get("steps", 0), case.get("chunk", 1)
    total = case["T"] + steps * chunk
    query, key = _logits(generator, (case["S"], total, case["H"], case["qk_bits"]), dtype,
                         case["pattern"])
    streams = [query, key, randn(case["S"], total, case["Hp"], case["payload_bits"])]
    if not case["logits"]:
        widths = (case["qk_bits"], case["qk_bits"], case["payload_bits"])
        streams = [_symbols(stream, bits) for stream, bits in zip(streams, widths)]
    bounds = [0, *range(case["T"], total + 1, chunk)]
    updates = [tuple(stream[:, begin:end].contiguous() for stream in streams)
               for begin, end in zip(bounds, bounds[1:])]
    runtime = rosa_soft_amd.RosaRuntime(case["H"], case["Hp"], case["qk_bits"],
                                        case["payload_bits"], case["W"])
    return dict(kind=kind, runtime=runtime, updates=updates, logits=case["logits"])


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def _apply(state):
    query, key, value = state["arguments"]
    if state["offsets"] is None:
        return rosa_soft_amd.rosa_soft(query, key, value, **state["controls"])
    return rosa_soft_amd.rosa_soft_varlen(query, key, value, state["offsets"],
                                          **state["controls"])


def run(state):
    kind = state["kind"]
    if kind == "train":
        if state["controls"]["dropout_p"] > 0:
            # a program that wants repeatable steps seeds the generator the mask is drawn from
            torch.cuda.manual_seed(state["seed"])
        output = _apply(state)
        gradients = torch.autograd.grad(output, state["arguments"], state["grad_output"])
        return [output.detach(), *gradients]
    if kind == "forward":
        with torch.no_grad():
            return _apply(state)
    if kind == "project":
        query, key, value = state["arguments"]
        sign_words, routed = cabi.hard_forward_bits(query, key, value, state["controls"])
        return cabi.project_routed_bits(sign_words, routed, state["value_dim"], state["weight"],
                                        state["residual"])
    runtime = state["runtime"]
    runtime.reset()
    update = runtime.update if state["logits"] else runtime.update_packed
    results = [update(*symbols) for symbols in state["updates"]]
    if len(results) == 1:
        return list(results[0])
    return [torch.cat([result[part] for result in results], dim=1) for part in (0, 1)]


# ---------------------------------------------------------------------------
# what a pass needs, and how exact it is
# ---------------------------------------------------------------------------

def work(case):
    kind, item = case["kind"], ITEM_BYTES[case["dtype"]]
    if kind in ("train", "forward", "project"):
        lengths = _lengths(case)
        tokens = sum(lengths)
        inputs = tokens * (2 * case["H"] * case["D"] + case["Hv"] * case["Dv"]) * item
        outputs = tokens * case["H"] * case["Dv"] * item
        if kind == "forward":
            return {"bytes": inputs + outputs, "flops": 0}
        if kind == "project":
            depth = case["H"] * case["Dv"]
            # the activation between the two steps need not exist as a tensor
            return {"bytes": inputs + (2 * tokens + depth) * case["N"] * item,
                    "flops": 2 * tokens * depth * case["N"]}
        # output, its gradient, the three inputs and their gradients; and the five causal
        # contractions of the surrogate: q.k, go.v, dV, dK, dQ
        pairs = case["H"] * sum(n * (n - 1) // 2 for n in lengths)
        return {"bytes": 2 * (inputs + outputs),
                "flops": 2 * pairs * (3 * case["D"] + 2 * case["Dv"])}
    tokens = case["S"] * (case["T"] + case.get("steps", 0) * case.get("chunk", 1))
    heads, payload_heads = case["H"], case["Hp"]
    if case["logits"]:
        inputs = 2 * heads * case["qk_bits"] + payload_heads * case["payload_bits"]
        return {"bytes": tokens * (inputs * item + heads * (case["payload_bits"] * item + 8)),
                "flops": 0}
    return {"bytes": tokens * (2 * heads + payload_heads + heads * (1 + 8)), "flops": 0}


def tolerance(case):
    if case["kind"] == "train":
        # float32: sums over routes in any order with hardware exp2 and rsq; the narrow types:
        # the same gradients rounded to the input's type
        return {"rel": {"float32": 3e-5, "float16": 1e-3, "bfloat16": 5e-3}[case["dtype"]]}
    if case["kind"] == "project":
        return {"rel": 5e-3}  # float32 sums of bfloat16 products, rounded to bfloat16
    return "exact"  # ternary outputs, symbols and positions
