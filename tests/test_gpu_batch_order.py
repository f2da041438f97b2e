"""Batches start in the order of descending key length: whatever the order, every slice has to be computed once.  As many
batches as are ranked and one more (64 / 65 with key lengths, 16 / 17 with a keep-mask of keys), equal lengths, an empty
sequence, two batches, against the CPU oracle, forward and backward."""
import numpy as np
import pytest
import torch

from flame_amd import workloads as W
from tests.gpu_util import assert_close_bf16, to_dev, to_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,kind,masked", [
    (2, 40, "ascending", False), (5, 16, "ties", False), (64, 2, "random", False), (65, 2, "random", False), (9, 8, "causal", False),
    (2, 40, "ascending", True), (5, 16, "ties", True), (16, 5, "random", True), (17, 5, "random", True)])
def test_against_the_oracle(oracle, B, H, kind, masked):
    from flame_amd import capi
    print(f"[batch order] {B=} {H=} {kind=} {masked=}", flush=True)
    Sq, Sk, D, causal = 130, 210, 64, kind == "causal"
    rng = np.random.default_rng(B)
    # Random lengths are 32 and above: an element of dK sums Sq products of q and dS, which is rounded to bf16, so its error is
    # about scale sqrt(Sq) |dP - delta| P 2^-9 / sqrt(3) = 0.125 * 11.4 * 8 * P * 1.1e-3 = 0.0125 P, and its largest over 2e6
    # elements five times that: 0.03 with two or three keys (P = 1 / 2), past the flat 2e-2 bar, and below 0.01 with 32.
    lens = {"ascending": np.arange(1, B + 1) * Sk // B, "ties": np.array([64, 200, 64, 0 if not masked else 1, 200])}.get(kind, rng.integers(32, Sk + 1, B))
    lens = lens.astype(np.int32)
    q, k, v, do = (W.f32_to_bf16_bits(W.normal_f32(7900 + B, s, B * H * n * D).reshape(B, H, n, D)) for s, n in enumerate((Sq, Sk, Sk, Sq)))
    sc = D ** -0.5
    ro, _, ro32 = oracle.sdpa_fwd(q, k, v, sc, causal=causal, kv_len=lens, want_f32=True)
    rg = oracle.sdpa_bwd(q, k, v, ro, do, sc, causal=causal, kv_len=lens, want_f32=True)
    kw = dict(mask=torch.from_numpy((np.arange(Sk)[None, :] < lens[:, None]).astype(np.uint8)).cuda().view(B, 1, 1, Sk)) if masked else \
        dict(kv_len=torch.from_numpy(lens).cuda(), causal=causal)
    dq_, dk_, dv_, do_ = (to_dev(t) for t in (q, k, v, do))
    o, lse = capi.attn_fwd(dq_, dk_, dv_, sc, **kw)
    grads = capi.attn_bwd(dq_, dk_, dv_, o, do_, lse, sc, **kw)
    torch.cuda.synchronize()
    assert_close_bf16(oracle, "O", to_f32(o), ro, ro32)
    for name, a, bits, f32 in zip(("dQ", "dK", "dV"), grads, rg[:3], rg[3:]):
        assert_close_bf16(oracle, name, to_f32(a), bits, f32)
