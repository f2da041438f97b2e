"""The dropout kernels that draw a tile row at a time (key counts that are multiples of 64) and those that draw element by
element, on grids large enough for the 128-query forward: the kept set bit for bit, read off O through a one-hot V, and
forward and backward against the CPU oracle; one key past a tile, an odd key count, several key tiles, padded head dims."""
import numpy as np
import pytest
import torch

from flame_amd import workloads as W
from tests.gpu_util import assert_close_bf16, to_dev, to_f32

pytestmark = pytest.mark.gpu
SEED = 0x2545F4914F6CDD1D
B, H = 3, 22        # 66 heads: more than a quarter of the compute units' worth of 128-query workgroups


@pytest.mark.parametrize("Sq,Sk,D,causal", [(130, 192, 64, False), (130, 191, 64, False), (70, 128, 128, True), (129, 65, 72, False)])
def test_kept_set_and_values(oracle, Sq, Sk, D, causal):
    from flame_amd import capi
    print(f"[dropout rows] {Sq=} {Sk=} {D=} {causal=}", flush=True)
    q, k, v, do = (W.f32_to_bf16_bits(W.normal_f32(7600 + Sk, s, B * H * n * D).reshape(B, H, n, D)) for s, n in enumerate((Sq, Sk, Sk, Sq)))
    sc = D ** -0.5
    p = float(np.quantile(oracle.dropout_uniforms(B, H, Sq, Sk, SEED), 0.3))
    keep = oracle.dropout_keep_mask(B, H, Sq, Sk, p, SEED).reshape(B, H, Sq, Sk).astype(bool)
    dq_, dk_, dv_, do_ = (to_dev(t) for t in (q, k, v, do))
    for c0 in range(0, Sk, D):                      # key c0 + d shows in output column d
        w = min(D, Sk - c0)
        one = torch.zeros((B, H, Sk, D), device="cuda", dtype=torch.bfloat16)
        one[:, :, c0 + torch.arange(w), torch.arange(w)] = 1.0
        o, _ = capi.attn_fwd_dropout(torch.zeros_like(dq_), dk_, one, sc, p, SEED)
        assert np.array_equal(to_f32(o)[..., :w] != 0, keep[..., c0:c0 + w])
    ro, rlse, ro32 = oracle.sdpa_fwd_dropout(q, k, v, sc, p, SEED, causal=causal, want_f32=True)
    o, lse = capi.attn_fwd_dropout(dq_, dk_, dv_, sc, p, SEED, causal=causal)
    assert_close_bf16(oracle, "O", to_f32(o), ro, ro32)
    rg = oracle.sdpa_bwd_dropout(q, k, v, ro, do, sc, p, SEED, causal=causal, want_f32=True)
    grads = capi.attn_bwd_dropout(dq_, dk_, dv_, to_dev(ro), do_, torch.from_numpy(rlse.reshape(B * H, Sq)).cuda(), sc, p, SEED, causal=causal)
    torch.cuda.synchronize()
    for name, a, bits, f32 in zip(("dQ", "dK", "dV"), grads, rg[:3], rg[3:]):
        assert_close_bf16(oracle, name, to_f32(a), bits, f32)
