"""Dropout backward on grids that leave compute units idle: key walks of dQ and query walks of dK/dV shared by several workgroups
(few heads), and the last round of the dK/dV key blocks split (30 heads: 14 key blocks beyond one per compute unit), for each
way of drawing, with causal and key lengths; against the CPU oracle and against the same call without room for partial sums."""
import numpy as np
import pytest
import torch

from flame_amd import workloads as W
from tests.gpu_util import assert_close_bf16, to_dev, to_f32

pytestmark = pytest.mark.gpu
SEED, P = 0x2545F4914F6CDD1D, 0.2


@pytest.mark.parametrize("B,H,Sq,Sk,D,causal,kv_len,chunks", [
    (1, 2, 1100, 1100, 64, False, None, (0, 0)), (1, 2, 1088, 1088, 128, True, None, (0, 0)), (2, 1, 1050, 1025, 72, False, [1025, 300], (0, 0)),
    (1, 1, 1100, 1088, 64, False, None, (512, 256)), (1, 30, 1040, 1100, 64, False, None, (0, 0)), (1, 30, 1040, 1152, 64, False, None, (0, 0))])
def test_shared_walks(oracle, B, H, Sq, Sk, D, causal, kv_len, chunks):
    from flame_amd import capi
    print(f"[dropout walks] {B=} {H=} {Sq=} {Sk=} {D=} {causal=} {kv_len=} {chunks=}", flush=True)
    q, k, v, do = (W.f32_to_bf16_bits(W.normal_f32(8100 + Sk, s, B * H * n * D).reshape(B, H, n, D)) for s, n in enumerate((Sq, Sk, Sk, Sq)))
    sc = D ** -0.5
    kw = dict(draw_chunk_q=chunks[0], draw_chunk_kv=chunks[1], causal=causal)
    dl = None if kv_len is None else torch.tensor(kv_len, dtype=torch.int32, device="cuda")
    dq_, dk_, dv_, do_ = (to_dev(t) for t in (q, k, v, do))
    o, lse = capi.attn_fwd_dropout(dq_, dk_, dv_, sc, P, SEED, kv_len=dl, **kw)
    got = capi.attn_bwd_dropout(dq_, dk_, dv_, o, do_, lse, sc, P, SEED, kv_len=dl, **kw)
    rows = torch.empty(2 * ((B * H * Sq * 4 + 255) // 256 * 256), dtype=torch.uint8, device="cuda")       # no room for partial sums
    alone = capi.attn_bwd_dropout(dq_, dk_, dv_, o, do_, lse, sc, P, SEED, kv_len=dl, workspace=rows, **kw)
    for name, a, b in zip(("dQ", "dK", "dV"), got, alone):
        # the same products, added up in another order in fp32: at most the last bit of bf16 differs, and rarely
        a, b = a.float(), b.float()
        assert float((a - b).abs().max()) <= 2 ** -7 * float(b.abs().max()), name
        assert float((a - b).norm()) <= 1e-3 * float(b.norm()), name
    bits = o.view(torch.uint16).cpu().numpy()
    rg = oracle.sdpa_bwd_dropout(q, k, v, bits, do, sc, P, SEED, causal=causal, kv_len=kv_len, want_f32=True, chunk_q=chunks[0], chunk_kv=chunks[1])
    for name, a, b, f32 in zip(("dQ", "dK", "dV"), got, rg[:3], rg[3:]):
        assert_close_bf16(oracle, name, to_f32(a), b, f32)
