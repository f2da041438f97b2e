"""The attention workloads whose speed is tracked: what each is, its inputs, one pass over it, and what it cannot do
without.  Every pass goes through the public Python interface (`flame_amd.functional`, `flame_amd.capi`) as a caller's
program does; sizes are those of the benchmark configurations and tests, or generic ones around them.

A case is a dict of plain values.  `kind` says what is called:

  train        functional.sdpa, forward and torch.autograd backward (optional causal flag, keep-mask)
  infer        functional.sdpa without gradients (optional causal flag, keep-mask); a few query rows against long keys too
  ragged       capi.attn_fwd + capi.attn_bwd with per-sequence key lengths
  bias         functional.sdpa_with_bias: additive fp32 relative-position bias, unscaled logits
  dropout      capi.attn_fwd_dropout + capi.attn_bwd_dropout
  joint_infer  capi.prep_rmsnorm_rope on the query and key projections, then functional.sdpa
  sage         capi.sage_quant + capi.sage_fwd (int8 QK^T)
  offload      capi.bf16_to_fp8 + capi.fp8_to_bf16 of the activations saved for the backward
"""
from __future__ import annotations

import math

import torch

from flame_amd import capi, functional, workloads

DEFAULTS = dict(B=1, H=1, Sq=256, Sk=256, D=64, causal=False, mask="none", dtype="bf16", layout="bhnd", p=0.0, text=0)


def _case(kind, **kw):
    return dict(DEFAULTS, kind=kind, **kw)


def listed():
    return [
        # the smallest training step (the benchmark's small configuration): launches and host time decide
        _case("train", name="train_small", B=1, H=4, Sq=256, Sk=256, D=64),
        # one training step of a diffusion transformer's joint text + image attention (the headline configuration)
        _case("train", name="train_dit_joint", B=1, H=24, Sq=4608, Sk=4608, D=128),
        # long causal self-attention, training: the largest problem
        _case("train", name="train_causal_long", B=1, H=32, Sq=16384, Sk=16384, D=128, causal=True),
        # training on a padded batch: a boolean key-padding mask [B, 1, 1, Sk], a length that is no multiple of a tile
        _case("train", name="train_padded_batch", B=4, H=16, Sq=1101, Sk=1101, D=128, mask="keys"),
        # training through one wide head, as in the mid block of an image autoencoder: head dim above 128
        _case("train", name="train_wide_head", B=1, H=1, Sq=4096, Sk=4096, D=512),
        # cross attention onto prompts of very different lengths, training, key lengths per sequence
        _case("ragged", name="train_ragged_cross", B=4, H=16, Sq=1024, Sk=2049, D=64),
        # training with dropout of the probabilities
        _case("dropout", name="train_dropout", B=2, H=16, Sq=1024, Sk=1024, D=64, p=0.1),
        # a text encoder with a relative-position bias (unscaled logits, inference)
        _case("bias", name="encoder_bias", B=1, H=64, Sq=512, Sk=512, D=64),
        # inference of the joint attention from the projections' [B, N, H, D] outputs: normalise + rotate Q and K, attend
        _case("joint_infer", name="joint_infer", B=2, H=24, Sq=1536, Sk=1536, D=128, layout="bnhd", text=512),
        # int8 QK^T inference at the benchmark's size
        _case("sage", name="int8_infer", B=2, H=24, Sq=4608, Sk=4608, D=128),
        # one new query row per sequence against the keys and values of all earlier ones
        _case("infer", name="decode_step", B=2, H=32, Sq=1, Sk=4097, D=128),
        # the saved activations of the headline layer (Q, K, V, O) to their FP8 form and back
        _case("offload", name="offload_fp8", B=1, H=24, Sq=4608, Sk=4608, D=128),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _length(rng, lo, hi):
    """A sequence length: half of them whole tiles of 64 (image grids, packed buffers), half as they come."""
    n = _log(rng, lo, hi)
    return max(64, n // 64 * 64) if rng.random() < 0.5 else n


def draw(rng):
    kind = rng.choice(["train", "train", "train_causal", "train_masked", "train_wide", "ragged", "dropout", "bias",
                       "joint_infer", "sage", "decode", "infer", "offload"])
    D = rng.choice([40, 64, 64, 72, 80, 96, 128, 128, 128])
    B, H = rng.randint(1, 4), rng.choice([1, 4, 8, 12, 16, 24, 30, 32])
    layout = rng.choice(["bhnd", "bnhd"])
    if kind == "train":                       # self and cross attention, small and large
        Sq = _length(rng, 64, 8192)
        Sk = Sq if rng.random() < 0.6 else _length(rng, 16, 4096)
        return _bounded(_case("train", B=B, H=H, Sq=Sq, Sk=Sk, D=D, layout=layout))
    if kind == "train_causal":
        S = _length(rng, 64, 16384)
        return _bounded(_case("train", B=B, H=H, Sq=S, Sk=S, D=D, causal=True, layout=layout))
    if kind == "train_masked":
        Sq = _length(rng, 128, 4096)
        Sk = Sq if rng.random() < 0.6 else _length(rng, 64, 2048)
        return _bounded(_case("train", B=B, H=H, Sq=Sq, Sk=Sk, D=D, mask=rng.choice(["keys", "keys", "rows"]), layout=layout))
    if kind == "train_wide":
        S = _length(rng, 256, 4096)
        return _bounded(_case("train", B=B, H=rng.choice([1, 1, 2, 4, 8]), Sq=S, Sk=S, D=rng.choice([160, 192, 256, 264, 320, 384, 512, 512]),
                              causal=rng.random() < 0.2, layout=layout))
    if kind == "ragged":
        return _bounded(_case("ragged", B=rng.randint(2, 8), H=H, Sq=_length(rng, 128, 4096), Sk=_length(rng, 77, 4096), D=D, layout=layout))
    if kind == "dropout":
        S = _length(rng, 128, 4096)
        return _bounded(_case("dropout", B=B, H=H, Sq=S, Sk=S, D=D, p=rng.choice([0.05, 0.1, 0.2]), causal=rng.random() < 0.3))
    if kind == "bias":
        S = _length(rng, 64, 2048)
        return _bounded(_case("bias", B=B, H=rng.choice([8, 12, 16, 32, 64]), Sq=S, Sk=S, D=rng.choice([64, 64, 128]), layout=layout))
    if kind == "joint_infer":
        side, text = rng.randint(8, 96), rng.choice([77, 128, 256, 512])
        return _bounded(_case("joint_infer", B=B, H=H, Sq=text + side * side, Sk=text + side * side, D=rng.choice([64, 128, 128]),
                              layout="bnhd", text=text))
    if kind == "sage":
        S = _length(rng, 256, 8192)
        return _bounded(_case("sage", B=B, H=H, Sq=S, Sk=S, D=rng.choice([64, 96, 128, 128]), causal=rng.random() < 0.2))
    if kind == "decode":                      # one or a few new rows against a long cache
        return _bounded(_case("infer", B=_log(rng, 1, 16), H=H, Sq=rng.choice([1, 1, 1, 4, 16]), Sk=_log(rng, 128, 32768), D=D, layout=layout))
    if kind == "infer":                       # encoders: 77-token prompts, image patches; some programs keep fp32 activations
        S = rng.choice([77, 197, 257, 577, _length(rng, 64, 8192)])
        return _bounded(_case("infer", B=B, H=H, Sq=S, Sk=S, D=D, causal=rng.random() < 0.4, layout=layout,
                              dtype=rng.choice(["bf16", "bf16", "f32"])))
    return _bounded(_case("offload", B=B, H=H, Sq=_length(rng, 64, 8192), Sk=64, D=D))


def _bounded(case):
    """Fewer heads where the drawn sizes together would cost more than the largest listed case."""
    most = 4e12 if case["D"] <= 128 else 1e12
    while case["H"] > 1 and 14.0 * case["B"] * case["H"] * case["Sq"] * case["Sk"] * case["D"] > most:
        case["H"] //= 2
    while case["B"] > 1 and 14.0 * case["B"] * case["H"] * case["Sq"] * case["Sk"] * case["D"] > most:
        case["B"] -= 1
    return case


# ---------------------------------------------------------------- inputs
def _randn(case, g, heads_first_shape, mul=1.0):
    """A [B, H, N, D] tensor, in memory either that order or a view of the projections' [B, N, H, D] order."""
    B, H, N, D = heads_first_shape
    dt = torch.float32 if case["dtype"] == "f32" else torch.bfloat16
    shape = (B, N, H, D) if case["layout"] == "bnhd" else (B, H, N, D)
    x = torch.randn(shape, device="cuda", dtype=torch.float32, generator=g)
    x = (x * mul if mul != 1.0 else x).to(dt)
    return x.permute(0, 2, 1, 3) if case["layout"] == "bnhd" else x


def _key_lengths(case, g):
    """One length per sequence, spread over (0, Sk], the longest being Sk."""
    B, Sk = case["B"], case["Sk"]
    n = (torch.rand((B,), device="cuda", generator=g) * Sk).ceil().clamp(1, Sk).to(torch.int32)
    n[-1] = Sk
    return n


def prepare(case, seed):
    c = dict(DEFAULTS, **case)
    g = torch.Generator(device="cuda").manual_seed(seed)
    B, H, Sq, Sk, D, kind = c["B"], c["H"], c["Sq"], c["Sk"], c["D"], c["kind"]
    s = dict(case=c, kind=kind, scale=1.0 / math.sqrt(D))
    if kind == "offload":
        s["saved"] = torch.randn((4, B, H, Sq, D), device="cuda", generator=g).to(torch.bfloat16)
        return s
    if kind == "joint_infer":
        side = int(round(math.sqrt(Sq - c["text"])))
        cos, sin = workloads.axial_rope_tables(c["text"], side, side, D)
        s["cos"], s["sin"] = torch.from_numpy(cos).cuda(), torch.from_numpy(sin).cuda()
        s["wq"], s["wk"] = ((1.0 + 0.1 * torch.randn((D,), device="cuda", generator=g)).to(torch.bfloat16) for _ in range(2))
        s["q"], s["k"] = (torch.randn((B, Sq, H, D), device="cuda", generator=g).to(torch.bfloat16) for _ in range(2))
        s["v"] = _randn(c, g, (B, H, Sk, D))
        return s
    q, k, v = _randn(c, g, (B, H, Sq, D)), _randn(c, g, (B, H, Sk, D)), _randn(c, g, (B, H, Sk, D))
    if kind == "sage":
        k[..., 7] = k[..., 7] * 3.0 + 1.5       # one outlier channel, as keys have
    if kind == "bias":
        q = q * (D ** -0.5)                     # the scale lives in the weights there: logits are used unscaled
        s["bias"] = torch.randn((1, H, Sq, Sk), device="cuda", generator=g)
    if kind in ("train", "ragged", "dropout"):
        s["do"] = _randn(c, g, (B, H, Sq, D))
    if kind == "ragged":
        s["kv_len"] = _key_lengths(c, g)
    s["mask"] = None
    if c["mask"] == "keys":
        s["mask"] = (torch.arange(Sk, device="cuda")[None, :] < _key_lengths(c, g)[:, None]).view(B, 1, 1, Sk)
    elif c["mask"] == "rows":                   # documents packed into one sequence attend to themselves
        cuts = torch.rand((B, 3), device="cuda", generator=g)
        doc = lambda n: (torch.arange(n, device="cuda")[None, :, None] / n >= cuts[:, None, :]).sum(-1)    # noqa: E731
        s["mask"] = (doc(Sq)[:, :, None] == doc(Sk)[:, None, :]).view(B, 1, Sq, Sk)
        s["mask"][..., 0] = True
    if kind == "dropout":
        s["p"], s["seed"] = c["p"], 1 + seed % (1 << 31)
    if kind == "train":
        q, k, v = (t.detach().requires_grad_(True) for t in (q, k, v))
    s["q"], s["k"], s["v"] = q, k, v
    return s


# ---------------------------------------------------------------- one pass
def run(s):
    c, kind = s["case"], s["kind"]
    if kind == "train":
        q, k, v = s["q"], s["k"], s["v"]
        o = functional.sdpa(q, k, v, attn_mask=s["mask"], is_causal=c["causal"])
        return (o, *torch.autograd.grad(o, (q, k, v), s["do"]))
    if kind == "infer":
        with torch.no_grad():
            return functional.sdpa(s["q"], s["k"], s["v"], attn_mask=s["mask"], is_causal=c["causal"])
    if kind == "ragged":
        o, lse = capi.attn_fwd(s["q"], s["k"], s["v"], s["scale"], kv_len=s["kv_len"])
        return (o, lse, *capi.attn_bwd(s["q"], s["k"], s["v"], o, s["do"], lse, s["scale"], kv_len=s["kv_len"]))
    if kind == "dropout":
        o, lse = capi.attn_fwd_dropout(s["q"], s["k"], s["v"], s["scale"], s["p"], s["seed"], causal=c["causal"])
        return (o, lse, *capi.attn_bwd_dropout(s["q"], s["k"], s["v"], o, s["do"], lse, s["scale"], s["p"], s["seed"], causal=c["causal"]))
    if kind == "bias":
        with torch.no_grad():
            return functional.sdpa_with_bias(s["q"], s["k"], s["v"], s["bias"], scale=1.0)
    if kind == "joint_infer":
        with torch.no_grad():
            q = capi.prep_rmsnorm_rope(s["q"], s["wq"], s["cos"], s["sin"])
            k = capi.prep_rmsnorm_rope(s["k"], s["wk"], s["cos"], s["sin"])
            return q, k, functional.sdpa(q, k, s["v"])
    if kind == "sage":
        z = capi.sage_quant(s["q"], s["k"])
        return z, capi.sage_fwd(z, s["v"], s["scale"], causal=c["causal"])
    codes = capi.bf16_to_fp8(s["saved"], 56.0)
    return codes, capi.fp8_to_bf16(codes, 1.0 / 56.0)


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    c = dict(DEFAULTS, **case)
    B, H, Sq, Sk, D, kind = c["B"], c["H"], c["Sq"], c["Sk"], c["D"], c["kind"]
    el = 4 if c["dtype"] == "f32" else 2
    nq, nk = B * H * Sq * D, B * H * Sk * D
    pairs = float(Sq) * Sk
    if c["causal"]:
        n = min(Sq, Sk)
        pairs = n * (n + 1) / 2.0 + float(Sq - n) * Sk
    pairs *= B * H
    if kind == "ragged" or c["mask"] == "keys":     # lengths are spread evenly, one sequence is full
        pairs *= (0.5 * (B - 1) + 1.0) / B
    if kind == "offload":
        n = 4 * nq
        return {"bytes": 6 * n, "flops": 0}
    if kind in ("train", "ragged", "dropout"):
        nbytes = el * (2 * nq + 2 * nk) + el * (nq + nq + 2 * nk)           # Q, K, V, dO in; O, dQ, dK, dV out
        flops = 14 * pairs * D
    else:
        nbytes = el * (nq + 2 * nk) + el * nq
        flops = 4 * pairs * D
    if kind == "joint_infer":
        nbytes += 2 * (nq + nk) + 8 * Sq * (D // 2) + 4 * D                 # the prepared Q and K come back too
    if kind == "sage":
        nbytes += nq + nk                                                   # the int8 codes come back too
    if kind == "bias":
        nbytes += 4 * H * Sq * Sk
    if c["mask"] == "keys":
        nbytes += B * Sk
    elif c["mask"] == "rows":
        nbytes += B * Sq * Sk
    if kind in ("ragged", "dropout"):
        nbytes += 4 * B * H * Sq                                            # the log-sum-exp comes back
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # FP8 codes and what they decode to are defined to the bit
    if case["kind"] == "offload":
        return "exact"
    # probabilities, dS and the outputs are bf16 (2^-9 each, of which the gradients chain three), sums are fp32
    return {"rel": 1e-2}
