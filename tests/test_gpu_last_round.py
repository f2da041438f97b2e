"""Grids of 256-query workgroups whose last round is cut into smaller workgroups in a launch of its own (32-query ones that share
the keys, or 128-query ones), forward and backward, against the CPU oracle: few left over with whole and with ragged query
tiles, and more left over than the key-sharing ones take."""
import pytest
import torch

from flame_amd import workloads as W
from tests.gpu_util import TOL_LSE, assert_close_bf16, to_dev, to_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("BH,Sq,Sk,D", [(130, 512, 64, 64), (130, 450, 128, 128), (180, 512, 64, 64), (130, 500, 64, 96)])
def test_against_the_oracle(oracle, BH, Sq, Sk, D):
    from flame_amd import capi
    print(f"[last round] {BH=} {Sq=} {Sk=} {D=}", flush=True)
    q, k, v, do = (W.f32_to_bf16_bits(W.normal_f32(7800 + D, s, BH * n * D).reshape(1, BH, n, D)) for s, n in enumerate((Sq, Sk, Sk, Sq)))
    sc = D ** -0.5
    ro, rlse, ro32 = oracle.sdpa_fwd(q, k, v, sc, want_f32=True)
    rg = oracle.sdpa_bwd(q, k, v, ro, do, sc, want_f32=True)
    dq_, dk_, dv_, do_ = (to_dev(t) for t in (q, k, v, do))
    o, lse = capi.attn_fwd(dq_, dk_, dv_, sc)
    grads = capi.attn_bwd(dq_, dk_, dv_, o, do_, lse, sc)
    torch.cuda.synchronize()
    assert_close_bf16(oracle, "O", to_f32(o), ro, ro32)
    assert abs(to_f32(lse).reshape(rlse.shape) - rlse).max() <= TOL_LSE
    for name, a, bits, f32 in zip(("dQ", "dK", "dV"), grads, rg[:3], rg[3:]):
        assert_close_bf16(oracle, name, to_f32(a), bits, f32)
