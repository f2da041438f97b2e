"""The 128-query forward and dQ kernels whose workgroups hold two groups of wavefronts with half of the key tiles each (one
workgroup per compute unit at most, 1024 keys or more, for dQ 2048): odd and even numbers of tiles, a ragged last tile, the second group
empty or without an attended key for some queries (causal, key lengths, an empty sequence), dropout by rows and by elements,
the largest grid that takes them and the next one, against the CPU oracle."""
import numpy as np
import pytest
import torch

from flame_amd import workloads as W
from tests.gpu_util import TOL_LSE, assert_close_bf16, to_dev, to_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,Sq,Sk,D,causal,lens,p", [
    (1, 130, 40, 1024, 64, False, None, 0.0), (1, 130, 40, 2050, 128, False, None, 0.0), (1, 131, 33, 2048, 72, False, None, 0.0),
    (1, 9, 2048, 2048, 128, True, None, 0.0), (2, 22, 300, 2100, 64, True, None, 0.0), (3, 44, 65, 2100, 64, False, (2100, 40, 0), 0.0),
    (1, 256, 20, 2049, 64, False, None, 0.0), (1, 257, 20, 2049, 64, False, None, 0.0), (1, 130, 40, 2048, 64, False, None, 0.2),
    (1, 130, 40, 2050, 128, False, None, 0.1), (1, 17, 1024, 1100, 64, True, None, 0.1)])
def test_forward_and_backward_against_the_oracle(oracle, B, H, Sq, Sk, D, causal, lens, p):
    from flame_amd import capi
    print(f"[key groups] {B=} {H=} {Sq=} {Sk=} {D=} {causal=} {lens=} {p=}", flush=True)
    q, k, v, do = (W.f32_to_bf16_bits(W.normal_f32(8100 + Sk, s, B * H * n * D).reshape(B, H, n, D)) for s, n in enumerate((Sq, Sk, Sk, Sq)))
    sc = D ** -0.5
    kvl = None if lens is None else np.asarray(lens, np.int32)
    dq_, dk_, dv_, do_ = (to_dev(t) for t in (q, k, v, do))
    if p:
        ro, rlse, ro32 = oracle.sdpa_fwd_dropout(q, k, v, sc, p, 77, causal=causal, want_f32=True)
        rg = oracle.sdpa_bwd_dropout(q, k, v, ro, do, sc, p, 77, causal=causal, want_f32=True)
        o, lse = capi.attn_fwd_dropout(dq_, dk_, dv_, sc, p, 77, causal=causal)
        grads = capi.attn_bwd_dropout(dq_, dk_, dv_, o, do_, lse, sc, p, 77, causal=causal)
    else:
        dkv = None if kvl is None else torch.from_numpy(kvl).cuda()
        ro, rlse, ro32 = oracle.sdpa_fwd(q, k, v, sc, causal=causal, kv_len=kvl, want_f32=True)
        rg = oracle.sdpa_bwd(q, k, v, ro, do, sc, causal=causal, kv_len=kvl, want_f32=True)
        o, lse = capi.attn_fwd(dq_, dk_, dv_, sc, causal=causal, kv_len=dkv)
        grads = capi.attn_bwd(dq_, dk_, dv_, o, do_, lse, sc, causal=causal, kv_len=dkv)
    torch.cuda.synchronize()
    assert_close_bf16(oracle, "O", to_f32(o), ro, ro32)
    got, fin = to_f32(lse).reshape(rlse.shape), np.isfinite(rlse)
    assert np.array_equal(fin, np.isfinite(got)) and np.abs(got[fin] - rlse[fin]).max(initial=0.0) <= TOL_LSE
    for name, a, bits, f32 in zip(("dQ", "dK", "dV"), grads, rg[:3], rg[3:]):
        assert_close_bf16(oracle, name, to_f32(a), bits, f32)
