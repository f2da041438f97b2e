"""Every form of the fused dropout kernels without a mask: compiled for head dims 64, 96 and 128, drawing tile by tile, element by
element and a tile row at a time, with one group of wavefronts per workgroup and with two; forward and backward against the CPU
oracle, the backward on the oracle's O and log-sum-exp.  The launches say that the form asked for is the one that ran."""
import numpy as np
import pytest
import torch

from flame_amd import workloads as W
from tests.gpu_util import TOL_LSE, assert_close_bf16, recorded_launches, to_dev, to_f32

pytestmark = pytest.mark.gpu
SEED, P = 0x2545F4914F6CDD1D, 0.2
B, H, SQ = 1, 130, 40        # more query tiles than half of the compute units: no shared walks, no 32-query workgroups
TILED, FLAT, ROWS = 1, 2, 3


@pytest.mark.parametrize("D,compiled", [(64, 64), (72, 96), (96, 96), (128, 128)])
@pytest.mark.parametrize("draw,Sk,groups", [(TILED, 200, 1), (FLAT, 195, 1), (ROWS, 192, 1), (TILED, 2112, 2), (FLAT, 2050, 2), (ROWS, 2048, 2)])
def test_against_the_oracle(oracle, D, compiled, draw, Sk, groups):
    from flame_amd import capi
    print(f"[dropout forms] {D=} {draw=} {Sk=} {groups=}", flush=True)
    q, k, v, do = (W.f32_to_bf16_bits(W.normal_f32(8300 + Sk + D, s, B * H * n * D).reshape(B, H, n, D)) for s, n in enumerate((SQ, Sk, Sk, SQ)))
    sc, chunks = D ** -0.5, (33, 150) if draw == TILED else (0, 0)
    ro, rlse, ro32 = oracle.sdpa_fwd_dropout(q, k, v, sc, P, SEED, want_f32=True, chunk_q=chunks[0], chunk_kv=chunks[1])
    rg = oracle.sdpa_bwd_dropout(q, k, v, ro, do, sc, P, SEED, want_f32=True, chunk_q=chunks[0], chunk_kv=chunks[1])
    tq, tk, tv, tdo, to = (to_dev(t) for t in (q, k, v, do, ro))
    tl = torch.from_numpy(np.ascontiguousarray(rlse)).cuda().reshape(B * H, SQ)
    kw = dict(draw_chunk_q=chunks[0], draw_chunk_kv=chunks[1])
    forward = lambda: capi.attn_fwd_dropout(tq, tk, tv, sc, P, SEED, **kw)                       # noqa: E731
    backward = lambda: capi.attn_bwd_dropout(tq, tk, tv, to, tdo, tl, sc, P, SEED, **kw)         # noqa: E731
    o, lse = forward()
    assert_close_bf16(oracle, "O", to_f32(o), ro, ro32)
    assert np.abs(to_f32(lse).reshape(rlse.shape) - rlse).max() <= TOL_LSE
    for name, a, bits, f32 in zip(("dQ", "dK", "dV"), backward(), rg[:3], rg[3:]):
        assert_close_bf16(oracle, name, to_f32(a), bits, f32)
    names = [name for call in (forward, backward) for name, _, _ in recorded_launches(call) if name.startswith(("fwd_kernel", "bwd_d"))]
    assert names == [f"fwd_kernel<{compiled}, 0, 4, {draw}, {groups}, false>", f"bwd_dq_kernel<{compiled}, 0, 4, {draw}, {groups}>",
                     f"bwd_dkdv_kernel<{compiled}, false, false, false, {draw}, false>"], names
