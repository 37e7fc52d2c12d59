"""The work whose speed counts: what a RetNet / POP-RetNet program has this library do, through the public entry points
of flash_pop_amd, over the range of sizes such programs use.

Five kinds of case, one public call sequence each:

  decode     one token of one layer: rotary embedding, recurrent step, per-head norm + gate (no gradients)
  prefill    the forward of fused_chunk_retention without gradients: a prompt goes in, outputs and the state come out
  train      fused_chunk_retention forward and backward
  pop        one POP layer step (context in blocks, one suffix per block boundary) forward and backward, either as the
             single call flash_pop_retention_with_suffixes or, `op` = "two", as the call sequence of an unchanged
             caller: flash_pop_retention, the states stacked, fused_chunk_retention on the suffix batch
  layer_ops  the elementwise stages next to the retention in a training step: rotary embedding of q and k, per-head norm
             + swish gate, both directions

Everything is bfloat16, the only type these entry points take.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "flash-pop_amd"))

from flash_pop_amd import (  # noqa: E402
    XPos, flash_pop_retention, flash_pop_retention_with_suffixes, fused_chunk_retention, gated_group_norm, retention_recurrent)

DIMS = ((64, 64), (64, 128), (128, 128), (128, 256))   # (dk, dv) of the configurations
HEADS = (4, 8, 12, 16)
TOKEN_HEADS = 8 * 4096 * 16                            # B * T * H of the largest training batch


def listed():
    return [
        # a chat-like loop: one sequence, every token a handful of tiny launches per layer; host and launch latency
        dict(name="decode_one", kind="decode", B=1, H=12, dk=64, dv=128, in_place=False),
        # a serving batch: 256 sequences, 134 MB of states read and written per layer and token
        dict(name="decode_batch", kind="decode", B=256, H=16, dk=128, dv=128, in_place=True),
        # a short prompt of a small model (B1 H4 T512 64 x 64)
        dict(name="prefill_short", kind="prefill", B=1, T=512, H=4, dk=64, dv=64, state=False),
        # one long prompt as it comes, no multiple of anything, continuing from a carried state
        dict(name="prefill_long", kind="prefill", B=1, T=5003, H=12, dk=64, dv=128, state=True),
        # the headline training shape
        dict(name="train_wide", kind="train", B=8, T=4096, H=16, dk=128, dv=128, state=False),
        # many small heads (B32 H4 T2048 64 x 64)
        dict(name="train_narrow", kind="train", B=32, T=2048, H=4, dk=64, dv=64, state=False),
        # a small batch of sequences cut where they end, truncated backpropagation: states carried in, their gradients out
        dict(name="train_ragged", kind="train", B=3, T=1777, H=8, dk=128, dv=128, state=True),
        # long context, few streams, wide values, states carried in and out
        dict(name="train_long", kind="train", B=2, T=16384, H=8, dk=128, dv=256, state=True),
        # POP world model at the headline shape: 64-token observations, 16 prediction tokens after each
        dict(name="pop_wide", kind="pop", op="one", B=8, T=4096, H=16, dk=128, dv=128, block=64, sfx=16),
        # one layer of the 12-layer POP decoder
        dict(name="pop_layer", kind="pop", op="one", B=8, T=2048, H=12, dk=64, dv=128, block=64, sfx=16),
        # an unchanged caller with observations of 144 tokens and 31 prediction tokens, ten observations per sequence
        dict(name="pop_two_calls", kind="pop", op="two", B=4, T=1440, H=4, dk=64, dv=128, block=144, sfx=31),
        # the elementwise stages of a training step at the headline shape
        dict(name="layer_ops", kind="layer_ops", B=8, T=4096, H=16, dk=128, dv=128),
    ]


def _log_int(rng, lo, hi):
    """An integer of lo .. hi, spread over the logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _length(rng, lo, hi):
    """A sequence length: half of them whole 64-token chunks, half as they come."""
    T = _log_int(rng, lo, hi)
    return max(64, T // 64 * 64) if rng.random() < 0.5 else T


def draw(rng):
    kind = rng.choice(("decode", "prefill", "prefill", "train", "train", "train", "pop", "pop", "layer_ops"))
    H = rng.choice(HEADS)
    dk, dv = rng.choice(DIMS)
    wide = (dk + dv) / 256                              # the budget of tokens is that of a 128 x 128 head
    if kind == "decode":
        return dict(kind=kind, B=_log_int(rng, 1, 256 if dk * dv * H <= 128 * 128 * 16 else 128), H=H, dk=dk, dv=dv,
                    in_place=rng.random() < 0.5)
    if kind == "pop":
        dk, dv = rng.choice(DIMS[:3])
        block = rng.choice((32, 64, 64, 64, 128, _log_int(rng, 15, 200)))
        sfx = rng.choice((16, 16, _log_int(rng, 1, 31)))
        T = block * max(2, _log_int(rng, 256, 4096) // block)
        op = rng.choice(("one", "two")) if block >= 64 else "one"
        B = _log_int(rng, 1, max(1, min(32, int((0.75 if op == "one" else 0.4) * TOKEN_HEADS / (T * (1 + sfx / block) * H)))))
        return dict(kind=kind, op=op, B=B, T=T, H=H, dk=dk, dv=dv, block=block, sfx=sfx)
    T = _length(rng, 64, 16384) if kind != "prefill" else _length(rng, 16, 16384)
    B = _log_int(rng, 1, max(1, min(64, int((0.8 if kind == "layer_ops" else 1.0) * TOKEN_HEADS / (T * H * max(wide, 0.5))))))
    if kind == "layer_ops":
        return dict(kind=kind, B=B, T=T, H=H, dk=dk, dv=dv)
    return dict(kind=kind, B=B, T=T, H=H, dk=dk, dv=dv, state=rng.random() < 0.5)


def _decays(H):
    return tuple(1.0 - 2.0 ** (-5.0 - h) for h in range(H))


def prepare(case, seed):
    B, H, dk, dv = case["B"], case["H"], case["dk"], case["dv"]
    T = case.get("T", 1)
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def randn(*shape, std=1.0):
        return (torch.randn(*shape, generator=gen, device="cuda") * std).to(torch.bfloat16)

    kind = case["kind"]
    st = dict(case, decays=_decays(H))
    st["q"], st["k"], st["v"] = randn(B, T, H, dk), randn(B, T, H, dk), randn(B, T, H, dv)
    if kind == "decode":
        st["s"], st["gate"], st["xpos"], st["pos"] = randn(B, H, dk, dv, std=0.3), randn(B, H * dv), XPos(dk), 1000 + seed % 1000
    elif kind == "layer_ops":
        st["gate"], st["xpos"] = randn(B, T, H * dv), XPos(dk)
        st["d_q"], st["d_k"], st["d_y"] = randn(B, T, H, dk), randn(B, T, H, dk), randn(B, T, H * dv)
        for name in ("q", "k", "v", "gate"):
            st[name].requires_grad_()
    elif kind == "pop":
        n = B * (T // case["block"] + 1)
        st["qs"], st["ks"], st["vs"] = (randn(n, case["sfx"], H, d) for d in (dk, dk, dv))
        st["s"] = torch.zeros(B, H, dk, dv, dtype=torch.bfloat16, device="cuda")
        st["d_o"], st["d_os"] = randn(B, T, H, dv), randn(n, case["sfx"], H, dv)
        for name in ("q", "k", "v", "qs", "ks", "vs"):
            st[name].requires_grad_()
    else:
        st["s"] = randn(B, H, dk, dv, std=0.02) if case["state"] else torch.zeros(B, H, dk, dv, dtype=torch.bfloat16, device="cuda")
        if kind == "train":
            st["d_o"] = randn(B, T, H, dv)
            st["leaves"] = [st["q"], st["k"], st["v"]]
            if case["state"]:
                st["d_s"] = randn(B, H, dk, dv)
                st["leaves"].append(st["s"])
            for t in st["leaves"]:
                t.requires_grad_()
    return st


def run(st):
    kind, decays = st["kind"], st["decays"]
    if kind == "decode":
        with torch.no_grad():
            q, k = st["xpos"](st["q"], st["k"], st["pos"])
            o, s = retention_recurrent(q[:, 0], k[:, 0], st["v"][:, 0], decays, st["s"], in_place=st["in_place"])
            return gated_group_norm(o, st["gate"]), s
    if kind == "prefill":
        with torch.no_grad():
            return fused_chunk_retention(st["q"], st["k"], st["v"], st["s"], decays)
    if kind == "train":
        o, s = fused_chunk_retention(st["q"], st["k"], st["v"], st["s"], decays)
        if st["state"]:
            grads = torch.autograd.grad([o, s], st["leaves"], [st["d_o"], st["d_s"]])
        else:
            grads = torch.autograd.grad([o], st["leaves"], [st["d_o"]])
        return o.detach(), s.detach(), grads
    if kind == "pop":
        ctx, sfx = (st["q"], st["k"], st["v"]), (st["qs"], st["ks"], st["vs"])
        if st["op"] == "one":
            o, o_s, last = flash_pop_retention_with_suffixes(*ctx, st["s"], decays, st["block"], *sfx)
        else:
            o, states = flash_pop_retention(*ctx, st["s"], decays, st["block"])
            starts = torch.cat((st["s"][:, None], states), dim=1).flatten(0, 1)
            o_s, _ = fused_chunk_retention(*sfx, starts, decays)
            last = states[:, -1]
        grads = torch.autograd.grad([o, o_s], ctx + sfx, [st["d_o"], st["d_os"]])
        return o.detach(), o_s.detach(), last.detach(), grads
    q, k = st["xpos"](st["q"], st["k"], 0)
    y = gated_group_norm(st["v"], st["gate"])
    grads = torch.autograd.grad([q, k, y], [st["q"], st["k"], st["v"], st["gate"]], [st["d_q"], st["d_k"], st["d_y"]])
    return q.detach(), k.detach(), y.detach(), grads


def work(case):
    """Bytes: every input once per direction and every output once (bf16); the states between the two calls of an
    unchanged POP caller are written and read, and so are their gradients.  Operations: the chunked form on dense 64-token
    tiles; a suffix token works on its suffix and reads one state."""
    B, H, dk, dv, T = case["B"], case["H"], case["dk"], case["dv"], case.get("T", 1)
    kind, n, mat = case["kind"], B * T * H, B * H * dk * dv
    if kind == "decode":
        return {"bytes": 2 * (B * H * (4 * dk + 4 * dv) + 2 * mat), "flops": 5 * mat}
    if kind == "layer_ops":
        return {"bytes": 2 * n * (8 * dk + 8 * dv), "flops": n * (12 * dk + 60 * dv)}

    def fwd_flops(tokens, C):
        return 2 * (C * (dk + dv) + 2 * dk * dv) * tokens

    def bwd_flops(tokens, C):
        return 2 * (C * (3 * dk + 2 * dv) + 4 * dk * dv) * tokens

    fwd_bytes, bwd_bytes = 2 * (2 * dk + 2 * dv), 2 * (4 * dk + 3 * dv)
    C = min(64, T)
    if kind == "prefill":
        return {"bytes": fwd_bytes * n + 2 * mat * (2 if case["state"] else 1), "flops": fwd_flops(n, C)}
    if kind == "train":
        return {"bytes": (fwd_bytes + bwd_bytes) * n + 2 * mat * (5 if case["state"] else 1), "flops": fwd_flops(n, C) + bwd_flops(n, C)}
    n_s = B * (T // case["block"] + 1) * case["sfx"] * H
    flops = fwd_flops(n, C) + bwd_flops(n, C) + (2 * (case["sfx"] * (dk + dv) + dk * dv) + 2 * (case["sfx"] * (3 * dk + 2 * dv) + 2 * dk * dv)) * n_s
    states = 4 * 2 * mat * (T // case["block"] + 1) if case["op"] == "two" else 0
    return {"bytes": (fwd_bytes + bwd_bytes) * (n + n_s) + 2 * mat + states, "flops": flops}


def tolerance(case):
    """Results are bf16 and the products inside take bf16 operands.  Against the same formulas in 64 bits (every kind, heads
    of slow and fast decay, up to 4096 tokens) the retention ops are off by at most 0.0034 (2-norm) and 0.034 (largest
    element); the elementwise stages, fp32 inside, by 0.0017 per rounding (0.0029 where two meet) and 0.010.  Four times
    what was seen; the decode chain ends in two roundings and an elementwise stage on a rounded sum."""
    return {"rel": 0.012, "max": 0.05} if case["kind"] in ("decode", "layer_ops") else {"rel": 0.013, "max": 0.14}
