"""The forward whose wavefronts share the keys of 32 queries (few query rows, few query tiles), against the CPU oracle at
the sizes where its tiling can go wrong: one row and the edges of the 32-query and 32-key tiles, walks shorter than its four
wavefronts, slices that get no key, key lengths that end inside another wavefront's tile, with and without room for a split."""
import math

import numpy as np
import pytest
import torch

from flame_amd import workloads as W
from tests.gpu_util import TOL_LSE, assert_close_bf16, to_dev, to_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,Sq,Sk,D,causal,lens", [
    (1, 2, 1, 1, 128, False, None), (2, 3, 1, 33, 64, False, None), (1, 1, 1, 4097, 128, False, None), (2, 2, 31, 127, 72, False, None),
    (1, 3, 32, 129, 128, True, None), (1, 2, 33, 128, 64, False, None), (1, 1, 65, 1000, 128, False, None), (3, 1, 16, 700, 40, False, (0, 65, 700)),
    (1, 2, 200, 200, 128, True, None), (2, 1, 4, 2049, 64, False, (1, 2049)), (1, 1, 96, 3000, 96, True, None)])
def test_against_the_oracle(oracle, B, H, Sq, Sk, D, causal, lens):
    from flame_amd import capi
    print(f"[keyshare] {B=} {H=} {Sq=} {Sk=} {D=} {causal=} {lens=}", flush=True)
    q, k, v = (W.f32_to_bf16_bits(W.normal_f32(7300 + Sk, s, B * H * n * D).reshape(B, H, n, D)) for s, n in enumerate((Sq, Sk, Sk)))
    sc = 1.0 / math.sqrt(D)
    kvl = None if lens is None else np.asarray(lens, np.int32)
    ro, rlse, ro32 = oracle.sdpa_fwd(q, k, v, sc, causal=causal, kv_len=kvl, want_f32=True)
    dq, dk, dv = (to_dev(t) for t in (q, k, v))
    dl = None if kvl is None else torch.from_numpy(kvl).cuda()
    for ws in (None, torch.empty(16, dtype=torch.uint8, device="cuda")):      # room as the call allocates it; too little for a split
        o, lse = capi.attn_fwd(dq, dk, dv, sc, causal=causal, kv_len=dl, workspace=ws)
        torch.cuda.synchronize()
        assert_close_bf16(oracle, "O", to_f32(o), ro, ro32)
        got, want = to_f32(lse).reshape(rlse.shape), rlse
        assert np.array_equal(np.isneginf(got), np.isneginf(want))
        fin = np.isfinite(want)
        assert np.abs(got[fin] - want[fin]).max(initial=0.0) <= TOL_LSE
