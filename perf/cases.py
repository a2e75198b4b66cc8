"""Workloads of this package for performance measurements.

Every case is one call of ``flash_attn_func`` on fp16 (batch, seqlen, heads, head_size)
tensors, as a user's program makes it: forward alone without autograd ("infer"), or
forward and backward through autograd ("train").  The package has no other direction:
queries and keys always have the same length.

Import with the repository's root as the working folder.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "flash-attention-v100_amd"))
from flash_attn_v100 import flash_attn_func  # noqa: E402


def _case(name, way, batch, heads, seqlen, dim, causal, scale=0.0, packed=False, padding=0):
    """way: "infer" or "train".  scale: softmax scale, 0 for the default 1/sqrt(dim).
    packed: q, k and v are slices of one (batch, seqlen, 3, heads, dim) projection output.
    padding: rows at the end of the sequence whose output the loss ignores (zero dout)."""
    return {"name": name, "way": way, "batch": batch, "heads": heads, "seqlen": seqlen, "dim": dim, "causal": causal,
            "scale": scale, "packed": packed, "padding": padding}


def listed():
    return [
        # a short text through a small encoder or decoder at batch 1: launches and host work are all there is
        _case("infer_b1_h8_n77_d64_causal", "infer", 1, 8, 77, 64, True),
        # the smallest training call: unit tests, tiny models, one attention layer of a toy run
        _case("train_b1_h4_n128_d64", "train", 1, 4, 128, 64, False),
        # BERT-base-shaped self-attention in training: many short sequences
        _case("train_b16_h12_n512_d64", "train", 16, 12, 512, 64, False),
        # GPT-style causal training at a short context
        _case("train_b4_h16_n1024_d64_causal", "train", 4, 16, 1024, 64, True),
        # prompt of one user, of no round length, with q, k and v straight from a fused projection
        _case("infer_b1_h32_n1500_d128_causal_packed", "infer", 1, 32, 1500, 128, True, packed=True),
        # bidirectional training on sequences cut at no multiple of anything, fused projection
        _case("train_b3_h20_n1031_d128_packed", "train", 3, 20, 1031, 128, False, packed=True),
        # long bidirectional encoder (documents, image patches) serving one input
        _case("infer_b1_h12_n8192_d64", "infer", 1, 12, 8192, 64, False),
        # causal training at a medium context with a scale of the caller's own
        _case("train_b2_h40_n2048_d128_causal", "train", 2, 40, 2048, 128, True, scale=0.1),
        # Llama-7B-shaped causal attention: prefill of two full contexts ...
        _case("infer_b2_h32_n4096_d128_causal", "infer", 2, 32, 4096, 128, True),
        # ... and a training step of the same
        _case("train_b2_h32_n4096_d128_causal", "train", 2, 32, 4096, 128, True),
        # long-context training, the last 32 rows being padding
        _case("train_b1_h16_n16384_d128_causal_padded", "train", 1, 16, 16384, 128, True, padding=32),
        # twice that length: the largest call
        _case("train_b1_h16_n32768_d128_causal", "train", 1, 16, 32768, 128, True),
    ]


def _pairs(case):
    """(query, key) pairs per (batch, head) slice that are not masked."""
    n = case["seqlen"]
    return n * (n + 1) // 2 if case["causal"] else n * n


def work(case):
    """Each input read once, each output written once; 2 matrix products forward, 5 backward."""
    rows = case["batch"] * case["heads"] * case["seqlen"]
    train = case["way"] == "train"
    tensors = 8 if train else 4  # q, k, v, o and dout, dq, dk, dv
    products = 7 if train else 2
    return {"bytes": tensors * rows * case["dim"] * 2,
            "flops": products * 2 * case["batch"] * case["heads"] * _pairs(case) * case["dim"]}


_MOST_FLOPS = 7 * 2 * 16 * (32768 * 32769 // 2) * 128  # of the largest listed case
_MOST_VALUES = 16 * 32768 * 128 * 2                    # of one tensor


def draw(rng):
    """Another call of the same ranges: 16 to 32768 positions, 1 to 16 sequences, 1 to 40 heads, both head sizes,
    masked or not, dense or packed, forward alone or forward and backward."""
    log_int = lambda lo, hi: int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))
    while True:
        case = {"way": rng.choice(["infer", "train"]), "batch": log_int(1, 16), "heads": log_int(1, 40),
                "seqlen": log_int(16, 32768), "dim": rng.choice([64, 128]), "causal": rng.random() < 0.6,
                "scale": 0.1 if rng.random() < 0.2 else 0.0, "packed": rng.random() < 0.3, "padding": 0}
        if case["way"] == "train" and case["seqlen"] >= 64 and rng.random() < 0.2:
            case["padding"] = rng.randint(1, 32)
        values = case["batch"] * case["heads"] * case["seqlen"] * case["dim"]
        if work(case)["flops"] <= _MOST_FLOPS and values <= _MOST_VALUES:
            return case


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    shape = (case["batch"], case["seqlen"], case["heads"], case["dim"])
    normal = lambda *s: torch.randn(s, device="cuda", dtype=torch.float16, generator=gen)
    if case["packed"]:
        q, k, v = normal(shape[0], shape[1], 3, shape[2], shape[3]).unbind(2)
    else:
        q, k, v = (normal(*shape) for _ in range(3))
    state = {"q": q, "k": k, "v": v, "scale": case["scale"] or None, "causal": case["causal"], "dout": None}
    if case["way"] == "train":
        state["dout"] = normal(*shape)
        if case["padding"]:
            state["dout"][:, -case["padding"]:] = 0
        for name in "qkv":
            state[name] = state[name].detach().requires_grad_()
    return state


def run(state):
    q, k, v, dout = state["q"], state["k"], state["v"], state["dout"]
    if dout is None:
        with torch.no_grad():
            return flash_attn_func(q, k, v, state["scale"], state["causal"])
    out = flash_attn_func(q, k, v, state["scale"], state["causal"])
    dq, dk, dv = torch.autograd.grad(out, (q, k, v), dout)
    return {"out": out, "dq": dq, "dk": dk, "dv": dv}


def tolerance(case):
    """fp16 results of fp32 sums over fp16 products: inputs, probabilities, dS and results carry relative roundings
    of 2^-11 each, and probabilities of long rows are fp16 subnormals (steps of 2^-24 where their mean is 2^-15)."""
    return {"rel": 2e-3}
