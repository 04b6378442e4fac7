"""The sampling calls whose time is followed, as a decode loop makes them: the two drop-in entry points
of the package over the range of batches, vocabularies, parameters and logit formats they serve.

A case is a dict of plain values:

  B, T, V      shape of the logits; T = 0: (B, V), else (B, T, V), of which the last position is sampled
  dtype        "float32", or "bfloat16" / "float16" (read as they are with accept_half=True)
  logits       "uniform" U[0,1) * scale, "normal" N(0,1) * scale, "spiked" N(0,1) * scale and +10 on 16 random
               tokens of each row (what a confident language model gives: a few candidates over a broad floor)
  scale        see logits
  temperature, top_k, top_p
  penalties    share of the (B, V) penalties that is non-zero (drawn from Exp(1)); 0: the call without penalties
"""
import torch

import rapid_sampling_amd as sample

# decay and the two penalties of the calls with penalties
PRESENCE, REPETITION, DECAY = 0.1, 0.1, 0.95

DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}


def _case(B, V, logits, scale, temperature, top_k, top_p, T=0, dtype="float32", penalties=0.0):
    return {"B": B, "T": T, "V": V, "dtype": dtype, "logits": logits, "scale": scale, "temperature": temperature,
            "top_k": top_k, "top_p": top_p, "penalties": penalties}


def listed():
    cases = [
        # a byte-level vocabulary: nothing but the call itself
        ("small_vocab", _case(16, 256, "normal", 2.0, 0.9, 40, 0.95)),
        # one user's decode loop, nucleus sampling on a peaked row of a large vocabulary
        ("one_row_nucleus", _case(1, 262144, "normal", 3.0, 1.0, -1, 0.3)),
        # the same on a flat row (an early checkpoint, a high temperature): the nucleus holds tens of thousands
        ("one_row_flat", _case(1, 131072, "uniform", 1.0, 1.0, -1, 0.5)),
        # a handful of users, a vocabulary that is no power of two and no whole number of slices
        ("few_rows_ragged", _case(13, 50260, "spiked", 2.0, 0.7, 40, 0.95)),
        # a serving batch with the usual top-k and top-p
        ("batch_topk", _case(64, 152064, "spiked", 2.0, 0.8, 50, 0.9)),
        # decode steps with presence and repetition penalties, decayed and updated in place
        ("decode_penalties", _case(32, 131072, "normal", 1.5, 0.8, 50, 0.9, penalties=0.02)),
        # a large serving batch, logits straight from a bfloat16 head
        ("batch_bf16", _case(256, 151936, "spiked", 2.0, 0.6, 20, 0.95, dtype="bfloat16")),
        # many rows, nucleus alone, half precision
        ("nucleus_fp16", _case(512, 32768, "normal", 3.0, 1.0, -1, 0.9, dtype="float16")),
        # plain temperature sampling: every token kept (rollouts for training)
        ("plain_temperature", _case(512, 50304, "normal", 2.0, 1.0, -1, 1.0)),
        # kept sets of thousands of tokens
        ("wide_nucleus", _case(128, 100256, "uniform", 4.0, 1.0, 10000, 0.9)),
        # a large batch with penalties
        ("large_penalties", _case(128, 262144, "normal", 1.5, 0.8, 50, 0.9, penalties=0.02)),
        # the last of several positions of the longest rows there are
        ("long_rows", _case(128, 1048576, "normal", 1.5, 1.0, 1024, 0.95, T=4)),
    ]
    return [dict(c, name=name) for name, c in cases]


def _log_uniform(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    """One more call: the kind of kept set, then a shape of that kind's range, odd sizes among them."""
    kind = rng.choice(["topk", "topk", "nucleus", "flat", "plain", "wide", "penalties", "penalties"])
    # tokens per call: up to 2^26, a quarter of that for the kinds that cost more per token
    most = 1 << (26 if kind in ("topk", "plain", "nucleus") else 24)
    V = 4 * _log_uniform(rng, 64, 262144)
    B = min(_log_uniform(rng, 1, 512), max(1, most // V))
    dtype = rng.choice(["float32", "float32", "bfloat16", "float16"])
    T = rng.choice([0, 0, 2]) if B * V <= 1 << 24 else 0
    temperature = round(rng.uniform(0.5, 1.3), 2)
    top_k, top_p, penalties = -1, round(rng.uniform(0.1, 0.95), 2), 0.0
    logits, scale = rng.choice([("normal", 3.0), ("spiked", 2.0), ("normal", 1.5)])
    if kind in ("topk", "penalties"):
        top_k = _log_uniform(rng, 1, min(1024, V))
        penalties = round(rng.uniform(0.001, 0.03), 4) if kind == "penalties" else 0.0
    elif kind == "plain":
        top_p = 1.0
    elif kind == "nucleus":
        logits, scale = rng.choice([("normal", 3.0), ("spiked", 2.0)])
    elif kind == "flat":
        logits, scale = rng.choice([("uniform", 1.0), ("uniform", 4.0), ("normal", 0.5)])
    else:
        top_k = min(V, _log_uniform(rng, 1025, 16384))
        logits, scale = rng.choice([("uniform", 4.0), ("normal", 1.5), ("normal", 0.5)])
    return _case(B, V, logits, scale, temperature, top_k, top_p, T=T, dtype=dtype, penalties=penalties)


def prepare(case, seed):
    B, T, V = case["B"], case["T"], case["V"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    shape = (B, T, V) if T else (B, V)
    if case["logits"] == "uniform":
        logits = torch.rand(shape, generator=gen, device="cuda").mul_(case["scale"])
    else:
        logits = torch.randn(shape, generator=gen, device="cuda").mul_(case["scale"])
    if case["logits"] == "spiked":
        rows = logits[:, T - 1] if T else logits
        where = torch.randint(0, V, (B, 16), generator=gen, device="cuda")
        rows.scatter_(1, where, rows.gather(1, where) + 10.0)
    penalties = None
    if case["penalties"]:
        penalties = torch.empty((B, V), device="cuda").exponential_(generator=gen)
        penalties.mul_(torch.rand((B, V), generator=gen, device="cuda") < case["penalties"])
    return {"logits": logits.to(DTYPES[case["dtype"]]), "penalties": penalties, "states": sample.setup_rand(seed, B),
            "temperature": case["temperature"], "top_k": case["top_k"], "top_p": case["top_p"],
            "accept_half": case["dtype"] != "float32"}


def run(state):
    """One decode step: the sampled tokens, and what the call updates in place."""
    if state["penalties"] is None:
        tokens = sample.batch_sampling_temperature_topk_topp(
            state["logits"], state["states"], state["temperature"], state["top_k"], state["top_p"],
            accept_half=state["accept_half"])
        return tokens, state["states"]
    tokens = sample.batch_sampling_repetition_temperature_topk_topp(
        state["logits"], state["penalties"], state["states"], PRESENCE, REPETITION, DECAY,
        state["temperature"], state["top_k"], state["top_p"], accept_half=state["accept_half"])
    return tokens, state["states"], state["penalties"]


def work(case):
    """Logits read once; penalties read and written once; per row the token and its generator state.
    Arithmetic per token: the scaling, the exponential (a degree-5 polynomial and its argument), a sum."""
    tokens = case["B"] * case["V"]
    size = 4 if case["dtype"] == "float32" else 2
    return {"bytes": tokens * (size + (8 if case["penalties"] else 0)) + case["B"] * (4 + 2 * sample.STATE_BYTES_PER_ROW),
            "flops": tokens * (16 + (3 if case["penalties"] else 0))}


def tolerance(case):
    """Every cross-token sum of the path is an exact integer and every floating-point step a single rounding:
    tokens, generator states and penalties are the same bits whatever the split of a row."""
    return "exact"
