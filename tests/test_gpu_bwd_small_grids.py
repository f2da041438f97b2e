"""Backward grids on at most half of the compute units, whose query walks (dK/dV) and key walks (dQ) are shared by several
workgroups and merged, against the CPU oracle: uneven shares, key lengths that leave shares and whole key blocks without a key
(one of them 0), a keep-mask of keys, causal with more keys than queries and the reverse, ragged tiles, padded head dims."""
import numpy as np
import pytest
import torch

from flame_amd import workloads as W
from tests.gpu_util import assert_close_bf16, to_dev, to_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,Sq,Sk,D,causal,lens,mask", [
    (1, 1, 1100, 1100, 64, False, None, False), (1, 2, 1031, 1990, 128, False, None, False), (1, 1, 1300, 900, 128, True, None, False),
    (1, 1, 900, 1500, 72, True, None, False), (3, 1, 1100, 1300, 64, False, (1300, 0, 70), False), (2, 1, 1090, 200, 128, False, None, True),
    (1, 1, 64, 2000, 128, False, None, False)])
def test_against_the_oracle(oracle, B, H, Sq, Sk, D, causal, lens, mask):
    from flame_amd import capi
    print(f"[bwd small grids] {B=} {H=} {Sq=} {Sk=} {D=} {causal=} {lens=} {mask=}", flush=True)
    q, k, v, do = (W.f32_to_bf16_bits(W.normal_f32(7900 + Sk, s, B * H * n * D).reshape(B, H, n, D)) for s, n in enumerate((Sq, Sk, Sk, Sq)))
    sc = D ** -0.5
    kvl = None if lens is None else np.asarray(lens, np.int32)
    m = None
    if mask:
        m = np.ones((B, 1, 1, Sk), np.uint8)
        m[0, ..., 100:] = 0
        m[1, ..., ::3] = 0
    full = None if m is None else np.ascontiguousarray(np.broadcast_to(m, (B, H, Sq, Sk)))
    ro, rlse = oracle.sdpa_fwd(q, k, v, sc, causal=causal, kv_len=kvl, mask=full)
    rg = oracle.sdpa_bwd(q, k, v, ro, do, sc, causal=causal, kv_len=kvl, mask=full, want_f32=True)
    grads = tuple(torch.full(t.shape, float("nan"), dtype=torch.bfloat16, device="cuda") for t in (q, k, v))
    capi.attn_bwd(*(to_dev(t) for t in (q, k, v, ro, do)), torch.from_numpy(np.ascontiguousarray(rlse).reshape(B * H, Sq)).cuda(), sc, causal=causal,
                  kv_len=None if kvl is None else torch.from_numpy(kvl).cuda(), mask=None if m is None else torch.from_numpy(m).cuda(), grads=grads)
    torch.cuda.synchronize()
    for name, a, bits, f32 in zip(("dQ", "dK", "dV"), grads, rg[:3], rg[3:]):
        assert_close_bf16(oracle, name, to_f32(a), bits, f32)
