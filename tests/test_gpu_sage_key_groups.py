"""The 128-query Sage forward whose workgroups hold two groups of wavefronts with half of the key tiles each (one workgroup per
compute unit at most, 1024 keys or more): odd and even numbers of tiles, a ragged last tile, the second group empty or without
an attended key for some queries (causal, key lengths), the short last round behind 256-query workgroups, K blocks scaled apart
so that a scale taken from another tile shows, against the CPU oracle on the same quantised operands."""
import numpy as np
import pytest

from flame_amd import workloads as W
from tests.gpu_util import TOL_LSE, assert_close_bf16, to_dev, to_f32

import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,Sq,Sk,D,causal,lens", [
    (1, 4, 130, 1024, 64, False, None), (1, 4, 130, 1090, 128, False, None), (1, 2, 1100, 1100, 64, True, None),
    (2, 2, 200, 1100, 128, False, (1100, 40)), (3, 2, 1030, 1100, 96, True, (1100, 600, 64)), (1, 33, 2048, 1088, 128, False, None)])
def test_against_the_oracle(oracle, B, H, Sq, Sk, D, causal, lens):
    from flame_amd import capi
    print(f"[sage key groups] {B=} {H=} {Sq=} {Sk=} {D=} {causal=} {lens=}", flush=True)
    qf, kf, vf = (W.normal_f32(8300 + Sk, s, B * H * n * D).reshape(B, H, n, D) for s, n in enumerate((Sq, Sk, Sk)))
    for jb in range(Sk // 64):
        kf[:, :, 64 * jb:64 * (jb + 1)] *= np.float32((1.0, 2.0, 0.25, 1.5, 0.5)[jb % 5])
    q, k, v = (W.f32_to_bf16_bits(t) for t in (qf, kf, vf))
    sc = float(0.5 / np.sqrt(D))
    z, ref = capi.sage_quant(to_dev(q), to_dev(k)), oracle.sage_quant(q, k)
    kvl = None if lens is None else np.asarray(lens, np.int32)
    o, lse = capi.sage_fwd(z, to_dev(v), sc, causal=causal, kv_len=None if kvl is None else torch.from_numpy(kvl).cuda(), want_lse=True)
    torch.cuda.synchronize()
    ro, rlse, ro32 = oracle.sage_fwd(ref["qi8"], ref["ki8"], ref["sq"], ref["sk"], v, sc, causal=causal, kv_len=kvl, want_f32=True)
    assert_close_bf16(oracle, "O", to_f32(o), ro, ro32)
    assert oracle.max_abs(lse.cpu().numpy().reshape(rlse.shape), rlse) <= TOL_LSE
