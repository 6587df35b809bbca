"""The work that a program has this package do, as cases that can be timed.

A case is one call of a public entry point: `EvoformerAttention.apply` (the reference's flat-reshape heads),
`DS4Sci_EvoformerAttention` (true heads), `evoformer_attention(..., gate=)` (the output gate) or
`GatedAttentionBlock` (the block around the attention).  `grad` says whether it is a training step (forward,
then the gradients of Q, K, V and the bias, or of everything the block has) or a forward without autograd, as in
inference.  Masks are what a crop pads away or drops: a bool keep-mask, or 0 / -1e9 added to the scores.
"""
from __future__ import annotations

import torch

from evoformer_triton_amd import DS4Sci_EvoformerAttention, EvoformerAttention, evoformer_attention
from evoformer_triton_amd.block import GatedAttentionBlock

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _case(entry, grad, dtype, shape, mask, bias, **more):
    B, S, N, H, D = shape
    return {"entry": entry, "grad": grad, "dtype": dtype, "B": B, "S": S, "N": N, "H": H, "D": D, "mask": mask, "bias": bias, **more}


def listed():
    return [
        # One short sequence without an alignment (the reference's first test shape), forward: the smallest call there is.
        dict(_case("flat", False, "bf16", (1, 1, 128, 16, 64), "bool", "fp32"), name="single-forward"),
        # A small fp32 training step (benchmark configuration C1): debugging and checks against other implementations.
        dict(_case("flat", True, "fp32", (1, 16, 64, 4, 32), "added", "same"), name="small-step-fp32"),
        # A fp32 training step of ordinary size, for those who do not train in 16 bits.
        dict(_case("flat", True, "fp32", (1, 64, 256, 8, 32), "added", "same"), name="msa-step-fp32"),
        # MSA row attention in training (C2, the headline configuration).
        dict(_case("flat", True, "bf16", (1, 512, 256, 8, 32), "added", "same"), name="msa-step"),
        # MSA row attention in inference: a protein's own length, gated, fp16, few alignment rows.
        dict(_case("gated", False, "fp16", (1, 128, 251, 8, 32), "added", "same"), name="msa-forward-ragged"),
        # Triangle attention in training (C3), through the DS4Sci calling convention.
        dict(_case("heads", True, "bf16", (1, 384, 384, 4, 32), "added", "same"), name="triangle-step"),
        # Triangle attention on a long crop (C4): the largest.
        dict(_case("flat", True, "bf16", (1, 768, 768, 4, 32), "added", "same"), name="triangle-step-long"),
        # Extra-MSA row attention with its small head dim (C5).
        dict(_case("flat", True, "bf16", (1, 1024, 384, 8, 8), "added", "same"), name="extra-msa-step"),
        # The shape family of the reference's speed benchmark: a batch of single sequences, many heads, fp32 bias.
        dict(_case("flat", True, "bf16", (4, 1, 1024, 32, 64), "bool", "fp32"), name="single-step-batch"),
        # The shape family of the reference's test matrix: head dim 64, fp32 bias, a few hundred rows.
        dict(_case("flat", True, "bf16", (1, 200, 640, 5, 64), "bool", "fp32"), name="rows-step-d64"),
        # Wide heads.
        dict(_case("heads", True, "bf16", (1, 64, 512, 4, 128), "added", "same"), name="rows-step-d128"),
        # The whole gated block in training: what a model's layer calls.
        dict(_case("block", True, "bf16", (1, 128, 256, 8, 32), "keep", "pair", c_m=256, c_z=128), name="block-step"),
    ]


def _spread(rng, lo, hi):
    """A whole number from lo to hi, evenly over the logarithm."""
    return max(lo, min(hi, round(lo * (hi / lo) ** rng.random())))


def _length(rng, lo, hi):
    """A row length: every other one as a crop has it (a multiple of 16), the others as a protein has it."""
    n = _spread(rng, lo, hi)
    return max(16, n // 16 * 16) if rng.random() < 0.5 else n


def draw(rng):
    kind = rng.choice(("single-forward", "step-fp32", "msa-step", "msa-forward", "triangle-step", "extra-msa-step", "single-step", "rows-d64",
                       "rows-d128", "block"))
    if kind == "single-forward":
        return _case("flat", False, "bf16", (rng.randint(1, 4), 1, _length(rng, 32, 512), rng.choice((4, 8, 16)), rng.choice((32, 64))), "bool", "fp32")
    if kind == "step-fp32":
        N = _length(rng, 32, 256)
        return _case("flat", True, "fp32", (1, _spread(rng, 4, max(4, 64 * 256 * 256 // (N * N) // 2)), N, rng.choice((4, 8)), 32), "added", "same")
    if kind == "msa-step":
        return _case(rng.choice(("flat", "heads")), True, rng.choice(("bf16", "bf16", "fp16")), (1, _spread(rng, 16, 512), _length(rng, 64, 384), 8, 32), "added", "same")
    if kind == "msa-forward":
        return _case("gated", False, rng.choice(("bf16", "fp16")), (1, _spread(rng, 8, 512), _length(rng, 64, 768), 8, 32), "added", "same")
    if kind == "triangle-step":
        N = _length(rng, 96, 768)
        return _case(rng.choice(("flat", "heads")), True, "bf16", (1, N, N, 4, 32), "added", "same")
    if kind == "extra-msa-step":
        return _case("flat", True, "bf16", (1, _spread(rng, 64, 1024), _length(rng, 96, 384), 8, 8), "added", "same")
    if kind == "single-step":
        return _case("flat", True, "bf16", (rng.randint(1, 4), 1, _length(rng, 128, 1024), 32, 64), "bool", "fp32")
    if kind == "rows-d64":
        return _case("flat", True, "bf16", (1, _spread(rng, 50, 200), _length(rng, 128, 768), rng.randint(1, 5), 64), "bool", "fp32")
    if kind == "rows-d128":
        return _case("heads", True, "bf16", (1, _spread(rng, 8, 64), _length(rng, 64, 512), 4, 128), "added", "same")
    return _case("block", True, "bf16", (1, _spread(rng, 16, 256), _length(rng, 64, 384), 8, 32), "keep", "pair", c_m=256, c_z=128)


def prepare(case, seed):
    B, S, N, H, D = (case[x] for x in "BSNHD")
    dt, dev = _DTYPES[case["dtype"]], torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(seed)

    def normal(*shape, dtype=dt):
        return torch.randn(shape, device=dev, generator=g).to(dtype)

    # Most residues stay: a crop's tail is padded (a length of its own per row) and some positions are dropped.
    tail = torch.randint(0, min(32, N // 4) + 1, (B, S, 1), device=dev, generator=g)
    keep = (torch.rand((B, S, N), device=dev, generator=g) < 0.95) & (torch.arange(N, device=dev) < N - tail)
    keep[:, :, 0] = True
    state = {"entry": case["entry"], "grad": case["grad"]}
    if case["entry"] == "block":
        with torch.random.fork_rng(devices=[dev]):
            torch.manual_seed(seed)
            block = GatedAttentionBlock(case["c_m"], D, H, c_z=case["c_z"], gating=True).to(dev).to(dt)
        m = normal(B, S, N, case["c_m"]).requires_grad_()
        z = normal(B, N, N, case["c_z"]).requires_grad_()
        state.update(block=block, m=m, z=z, mask=keep.float(), dout=normal(B, S, N, case["c_m"]), leaves=[m, z, *block.parameters()])
        return state
    q, k, v = (normal(B, S, N, H, D) for _ in range(3))
    bias = normal(B, 1, H, N, N, dtype=torch.float32 if case["bias"] == "fp32" else dt)
    mask = keep.view(B, S, 1, 1, N)
    if case["mask"] == "added":
        mask = torch.where(mask, 0.0, -1e9).to(dt)
    state.update(q=q, k=k, v=v, mask=mask, bias=bias)
    if case["entry"] == "gated":
        state["gate"] = normal(B, S, N, H, D)
    if case["grad"]:
        state["leaves"] = [q.requires_grad_(), k.requires_grad_(), v.requires_grad_(), bias.requires_grad_()]
        state["dout"] = normal(B, S, N, H, D)
    return state


def _forward(s):
    if s["entry"] == "block":
        return s["block"](s["m"], s["z"], s["mask"])
    if s["entry"] == "heads":
        return DS4Sci_EvoformerAttention(s["q"], s["k"], s["v"], [s["mask"], s["bias"]])
    if s["entry"] == "gated":
        return evoformer_attention(s["q"], s["k"], s["v"], s["mask"], s["bias"], layout="ds4sci", gate=s["gate"])
    return EvoformerAttention.apply(s["q"], s["k"], s["v"], s["mask"], s["bias"])


def run(state):
    if not state["grad"]:
        with torch.no_grad():
            return [_forward(state)]
    out = _forward(state)
    return [out, *torch.autograd.grad(out, state["leaves"], state["dout"])]


def work(case):
    """Each input read once, each output written once; two matrix products per score forward, five more backward."""
    B, S, N, H, D = (case[x] for x in "BSNHD")
    es = 4 if case["dtype"] == "fp32" else 2
    t, scores = B * S * N * H * D, B * S * H * N * N
    flops = (14 if case["grad"] else 4) * scores * D
    if case["entry"] == "block":
        c_m, c_z, hd = case["c_m"], case["c_z"], H * D
        rows, pairs = B * S * N, B * N * N
        weights = 5 * c_m * hd + c_z * H + hd + 3 * c_m + 2 * c_z
        flops += (6 if case["grad"] else 2) * (rows * c_m * hd * 5 + pairs * c_z * H)
        read, written = rows * c_m + pairs * c_z + weights, rows * c_m
        if case["grad"]:
            written += read
            read += rows * c_m
        return {"bytes": es * (read + written) + 4 * B * S * N, "flops": flops}
    bias = B * H * N * N * (4 if case["bias"] == "fp32" else es)
    mask = B * S * N * (1 if case["mask"] == "bool" else es)
    tensors = (8 if case["grad"] else 4) + (case["entry"] == "gated")
    return {"bytes": tensors * t * es + (2 if case["grad"] else 1) * bias + mask, "flops": flops}


def tolerance(case):
    """fp32: sums of up to some thousand fp32 terms; 16 bits: operands, P and dS rounded once each, and results rounded to 8 or 11 bits."""
    return {"rel": 1e-5, "max": 1e-3} if case["dtype"] == "fp32" else {"rel": 1e-2}
