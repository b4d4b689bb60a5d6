"""The attention calls that this package's speed is judged by, as plain data, and how to run one of them.

A case is one call of ``flex_attention`` (forward only), or one forward and backward (``train``) as a training step
makes it.  ``listed()`` holds the fixed cases, ``draw()`` one more of the same ranges; ``prepare()`` makes what a
program holds before the call, ``run()`` makes the call.
"""
import math

import torch

import flex_attention_tpu_amd as F
from flex_attention_tpu_amd import configs, masks, scores

WINDOW = 1025       # keys that a query of the windowed cases sees, its own among them
CAP = 30.0          # soft-cap of the logits
PREFIX = 96         # keys that every query of a prefix language model sees
CLOSURE_HEADS = 4   # heads that the position-bias closure's slopes are written for


def symmetric_alibi(s, b, h, q_idx, kv_idx):
    """A distance penalty on both sides of the query, a score function of a user's own."""
    return s - 2.0 ** (-8.0 * (h + 1) / 4) * torch.abs(q_idx - kv_idx)


def prefix_lm(q_idx, k_idx):
    """Causal behind a prefix that everyone sees, a mask of a user's own."""
    return (q_idx[:, None] >= k_idx[None, :]) | (k_idx[None, :] < PREFIX)


def _case(name=None, *, dtype="bf16", B, Hq, Hkv=None, Sq, Sk=None, D=128, mask="none", score="none", bias=False, train=True):
    c = dict(dtype=dtype, B=B, Hq=Hq, Hkv=Hkv or Hq, Sq=Sq, Sk=Sk or Sq, D=D, mask=mask, score=score, bias=bias, train=train)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest training step: float32, four heads, no mask; bound by launches and by the host
        _case("fp32_512_d64", dtype="fp32", B=1, Hq=4, Sq=512, D=64),
        # the short end of the sequence sweep (one sequence, eight heads): too little work to fill the chip by tiles
        _case("train_causal_1k", B=1, Hq=8, Sq=1024, mask="causal"),
        # one step of token generation: a query per sequence against a key cache of some thousand tokens
        _case("decode_6k", B=8, Hq=32, Hkv=8, Sq=1, Sk=6001, train=False),
        # a prompt of odd length read in before generation, grouped heads
        _case("prefill_2777", B=1, Hq=32, Hkv=8, Sq=2777, mask="causal", train=False),
        # the training step that the benchmark times
        _case("train_causal_4k", B=4, Hq=32, Sq=4096, mask="causal"),
        # sliding window with a position bias per head
        _case("train_alibi_window_8k", B=2, Hq=16, Sq=8192, mask="window", score="alibi"),
        # packed documents with capped logits and grouped heads
        _case("train_docs_softcap_16k", B=1, Hq=32, Hkv=8, Sq=16384, mask="document", score="softcap"),
        # narrow heads, as smaller models have them
        _case("train_causal_2k_d64", B=8, Hq=16, Sq=2048, D=64, mask="causal"),
        # wide heads
        _case("train_causal_4k_d256", B=4, Hq=16, Sq=4096, D=256, mask="causal"),
        # an encoder of odd length with a learned bias on the logits, shared by the batch
        _case("train_bias_1500", B=4, Hq=16, Sq=1500, bias=True),
        # a score function of the user's own, compiled into the kernels
        _case("train_closure_2k", B=8, Hq=CLOSURE_HEADS, Sq=2048, score="closure"),
        # the long end: one sequence of 64k tokens
        _case("train_causal_64k", B=1, Hq=8, Sq=65536, mask="causal"),
    ]


def _pairs(case):
    """Unmasked (query, key) pairs per head; a causal mask counts half of the square."""
    Sq, Sk = case["Sq"], case["Sk"]
    if case["mask"] == "window":
        return float(sum(min(i + 1, WINDOW) for i in range(Sq)))
    if case["mask"] == "document":
        return float(sum(n * (n + 1) // 2 for n in configs.segment_lengths(Sq)))
    if case["mask"] == "causal":
        return Sq * Sk / 2.0
    if case["mask"] == "prefix_lm":
        return Sq * Sk / 2.0 + PREFIX * min(PREFIX, Sq) / 2.0
    return float(Sq) * Sk


def work(case):
    size = 4 if case["dtype"] == "fp32" else 2
    B, Hq, Hkv, Sq, Sk, D = (case[n] for n in ("B", "Hq", "Hkv", "Sq", "Sk", "D"))
    rows, keys = B * Hq * Sq * D * size, B * Hkv * Sk * D * size
    plane = Hq * Sq * Sk * 4 if case["bias"] else 0
    flops = 4.0 * B * Hq * D * _pairs(case)
    nbytes = 2 * rows + 2 * keys + plane                  # q, k, v, the bias in; o out
    if case["train"]:
        flops *= 3.5                                      # five products behind the forward's two
        nbytes += 2 * rows + 2 * keys + plane             # do in; dq, dk, dv and the bias gradient out
    return {"bytes": nbytes, "flops": flops}


def _length(rng, lo, hi):
    """A sequence length, even over the logarithm of the range; half of them multiples of 128, the others anything."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(128, n // 128 * 128) if rng.random() < 0.5 else n


def draw(rng):
    kind = rng.choice(("fp32", "causal", "decode", "prefill", "alibi", "document", "d64", "d256", "bias", "closure"))
    most = max(work(c)["flops"] for c in listed())
    while True:
        B, groups, Hkv = rng.choice((1, 1, 2, 3, 4, 8)), rng.choice((1, 1, 2, 4, 8)), rng.choice((1, 2, 4, 6, 8, 16))
        Hq = Hkv * groups
        heads = dict(B=B, Hq=Hq, Hkv=Hkv)
        if kind == "fp32":
            c = _case(dtype="fp32", Sq=_length(rng, 128, 4096), D=rng.choice((64, 128)), mask=rng.choice(("none", "causal")), **heads)
        elif kind == "causal":
            c = _case(Sq=_length(rng, 512, 65536), mask="causal", score=rng.choice(("none", "none", "softcap")), **heads)
        elif kind == "decode":
            heads["B"] = rng.choice((1, 2, 4, 8, 16, 32))
            c = _case(Sq=rng.choice((1, 1, 1, 2, 5, 16)), Sk=_length(rng, 256, 32768), D=rng.choice((64, 128, 128)), train=False, **heads)
        elif kind == "prefill":
            c = _case(Sq=_length(rng, 200, 32768), mask="causal", train=False, **heads)
        elif kind == "alibi":
            c = _case(Sq=_length(rng, 512, 16384), mask=rng.choice(("window", "causal")), score="alibi", B=B, Hq=Hq)
        elif kind == "document":
            c = _case(Sq=_length(rng, 2048, 32768), mask="document", score=rng.choice(("none", "softcap")), **heads)
        elif kind == "d64":
            c = _case(Sq=_length(rng, 256, 16384), D=64, mask=rng.choice(("none", "causal", "causal")), **heads)
        elif kind == "d256":
            c = _case(Sq=_length(rng, 512, 16384), D=256, mask=rng.choice(("causal", "causal", "none")), **heads)
        elif kind == "bias":
            c = _case(Sq=_length(rng, 128, 2048), bias=True, B=B, Hq=Hq)
        elif rng.random() < 0.5:
            c = _case(Sq=_length(rng, 256, 8192), score="closure", B=B, Hq=CLOSURE_HEADS)
        else:
            c = _case(Sq=_length(rng, 256, 8192), mask="prefix_lm", **heads)
        w = work(c)
        if w["flops"] <= most / (40 if c["dtype"] == "fp32" else 2) and w["bytes"] < 8e9 and B * Hq <= 256:
            return c


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dtype = torch.float32 if case["dtype"] == "fp32" else torch.bfloat16
    B, Hq, Hkv, Sq, Sk, D = (case[n] for n in ("B", "Hq", "Hkv", "Sq", "Sk", "D"))
    train = case["train"]

    def normal(*shape, grad=False):
        return torch.randn(*shape, generator=g, device="cuda", dtype=dtype).requires_grad_(grad)
    state = {"q": normal(B, Hq, Sq, D, grad=train), "k": normal(B, Hkv, Sk, D, grad=train), "v": normal(B, Hkv, Sk, D, grad=train)}
    state["do"] = normal(B, Hq, Sq, D) if train else None
    state["ab"] = None
    if case["bias"]:   # (kept in float32, as a trained parameter is)
        state["ab"] = torch.randn(1, Hq, Sq, Sk, generator=g, device="cuda").requires_grad_(train)
    mask = {"none": lambda: None,
            "causal": lambda: masks.make_causal_mask_fns(128, 128),
            "window": lambda: masks.make_causal_sliding_window_mask_fns(128, 128, WINDOW),
            "document": lambda: masks.make_jagged_mask_fns(128, 128, configs.segment_lengths(Sq, seed=seed)),
            "prefix_lm": lambda: prefix_lm}[case["mask"]]()
    score = {"none": lambda: None,
             "alibi": lambda: scores.make_alibi_global_score_fn(Hq),
             "softcap": lambda: scores.make_softcap_score_fn(CAP),
             "closure": lambda: symmetric_alibi}[case["score"]]()
    state["args"] = (score, mask)
    # (a score function sees the products unscaled where the reference's drivers use one; 1 / sqrt(D) keeps them in range)
    state["sm_scale"] = 1.0 / math.sqrt(D)
    return state


def run(state):
    q, k, v, ab = state["q"], state["k"], state["v"], state["ab"]
    if state["do"] is None:
        with torch.no_grad():
            return F.flex_attention(q, k, v, *state["args"], sm_scale=state["sm_scale"])
    o = F.flex_attention(q, k, v, *state["args"], sm_scale=state["sm_scale"], ab=ab)
    wanted = (q, k, v) if ab is None else (q, k, v, ab)
    return (o.detach(), *torch.autograd.grad(o, wanted, state["do"]))


def tolerance(case):
    """About four times what the results differ by from the same computation in 64 bits: bfloat16 2.0e-3 to 3.0e-3
    (largest difference 0.1 of a value or of the root mean square), float32 3.5e-7 to 7e-7 (1.2e-5)."""
    if case["dtype"] == "fp32":
        return {"rel": 3e-6, "max": 5e-5}
    return {"rel": 1e-2, "max": 0.4}
