"""The key-sharing forward with eight wavefronts per workgroup (at most one workgroup per compute unit) and with four (more):
the edges of a round of 32-key tiles over the wavefronts, the head dims it is compiled for, and its three ways to draw a dropout,
against the CPU oracle."""
import math

import numpy as np
import pytest
import torch

from flame_amd import workloads as W
from tests.gpu_util import TOL_LSE, assert_close_bf16, recorded_launches, to_dev, to_f32

pytestmark = pytest.mark.gpu


def make(B, H, Sq, Sk, D):
    return [W.f32_to_bf16_bits(W.normal_f32(8800 + Sk + D, s, B * H * n * D).reshape(B, H, n, D)) for s, n in enumerate((Sq, Sk, Sk))]


def check(oracle, o, lse, ref):
    ro, rlse, ro32 = ref
    torch.cuda.synchronize()
    assert_close_bf16(oracle, "O", to_f32(o), ro, ro32)
    got = to_f32(lse).reshape(rlse.shape)
    assert np.array_equal(np.isneginf(got), np.isneginf(rlse))
    fin = np.isfinite(rlse)
    assert np.abs(got[fin] - rlse[fin]).max(initial=0.0) <= TOL_LSE


@pytest.mark.parametrize("B,H,Sq,Sk,D,causal,lens,compiled,waves", [
    (1, 2, 3, 255, 64, False, None, 64, 8), (1, 2, 33, 256, 96, True, None, 96, 8), (2, 1, 5, 257, 128, False, (256, 225), 128, 8),
    (1, 1, 31, 513, 72, False, None, 96, 8), (1, 4, 40, 289, 80, False, None, 96, 8), (1, 256, 2, 33, 64, False, None, 64, 8),
    (1, 257, 2, 127, 64, False, None, 64, 4), (2, 130, 1, 128, 128, False, (128, 1), 128, 4), (1, 260, 4, 161, 88, True, None, 96, 4)])
def test_wavefronts(oracle, B, H, Sq, Sk, D, causal, lens, compiled, waves):
    from flame_amd import capi
    print(f"[keyshare waves] {B=} {H=} {Sq=} {Sk=} {D=} {causal=} {lens=}", flush=True)
    q, k, v = make(B, H, Sq, Sk, D)
    sc = 1.0 / math.sqrt(D)
    kvl = None if lens is None else np.asarray(lens, np.int32)
    dq, dk, dv = (to_dev(t) for t in (q, k, v))
    dl = None if kvl is None else torch.from_numpy(kvl).cuda()
    few = torch.empty(16, dtype=torch.uint8, device="cuda")         # no room to split the keys

    def call():
        return capi.attn_fwd(dq, dk, dv, sc, causal=causal, kv_len=dl, workspace=few)
    check(oracle, *call(), oracle.sdpa_fwd(q, k, v, sc, causal=causal, kv_len=kvl, want_f32=True))
    (name, _, lanes), = recorded_launches(call)
    assert name.startswith(f"fwd_keyshare_kernel<{compiled}, {waves},") and lanes == 64 * waves, (name, lanes)


# rows that start on multiples of 64 elements, others, and a draw per 48 x 40 tile; more than 256 workgroups too
@pytest.mark.parametrize("B,H,Sq,Sk,D,causal,chunk", [
    (1, 3, 70, 320, 64, False, None), (1, 2, 64, 192, 96, True, None), (1, 3, 70, 301, 128, True, None), (1, 2, 100, 90, 40, False, None),
    (1, 2, 100, 90, 128, False, (48, 40)), (1, 258, 3, 128, 64, False, None), (1, 2, 100, 90, 64, True, (48, 40)), (1, 258, 3, 128, 64, False, (2, 64))])
def test_dropout(oracle, B, H, Sq, Sk, D, causal, chunk):
    from flame_amd import capi
    seed, sc = 0x2545F4914F6CDD1D, 1.0 / math.sqrt(D)
    print(f"[keyshare dropout] {B=} {H=} {Sq=} {Sk=} {D=} {causal=} {chunk=}", flush=True)
    q, k, v = make(B, H, Sq, Sk, D)
    cq, ck = chunk or (0, 0)
    p = float(np.quantile(oracle.dropout_uniforms(B, H, Sq, Sk, seed, cq, ck), 0.25))
    o, lse = capi.attn_fwd_dropout(*(to_dev(t) for t in (q, k, v)), sc, p, seed, causal=causal, draw_chunk_q=cq, draw_chunk_kv=ck)
    check(oracle, o, lse, oracle.sdpa_fwd_dropout(q, k, v, sc, p, seed, causal=causal, want_f32=True, chunk_q=cq, chunk_kv=ck))


# the largest logit among the keys of either half of a wavefront (keys 0 .. 3 of every eight, keys 4 .. 7), hundreds above all
# others: the maximum in use has to be that of both
@pytest.mark.parametrize("Sk,key", [(64, 6), (64, 33), (300, 299), (300, 260)])
def test_one_key_dominates(oracle, Sk, key):
    from flame_amd import capi
    print(f"[keyshare waves] {Sk=} {key=}", flush=True)
    q, k, v = make(1, 2, 5, Sk, 64)
    q[..., 0], k[..., 0] = W.f32_to_bf16_bits(np.float32([40.0])), 0
    k[:, :, key, 0] = W.f32_to_bf16_bits(np.float32([80.0]))
    o, lse = capi.attn_fwd(*(to_dev(t) for t in (q, k, v)), 0.125)
    check(oracle, o, lse, oracle.sdpa_fwd(q, k, v, 0.125, want_f32=True))
