"""The forward for head dims above 256 in two matrix products (taken where the caller, here the native host path, has room for
the probabilities): partial tiles of queries, keys and head dim, causal flag, key lengths (none, part of a tile, whole tiles
left out, with NaN in the keys and values past them), the split of the keys, several launches; against the CPU oracle or an fp32
reference.  A workspace too small for it means the one-pass kernel, which the other tests of these head dims hold to the oracle."""
import ctypes
import math

import numpy as np
import pytest
import torch

from flame_amd import workloads as W
from tests.gpu_util import TOL_LSE, assert_close_bf16, to_dev, to_f32

pytestmark = pytest.mark.gpu


def _inputs(seed, B, H, Sq, Sk, D):
    return [W.f32_to_bf16_bits(W.normal_f32(seed, s, B * H * n * D).reshape(B, H, n, D)) for s, n in enumerate((Sq, Sk, Sk))]


def _scratch(B, H, Sq, Sk, D):
    from flame_amd import capi
    f = capi.lib().flame_attn_fwd_scratch_bytes
    f.restype = ctypes.c_size_t
    return f(B, H, Sq, Sk, D), capi.fwd_workspace_bytes(B, H, Sq, Sk, D)


@pytest.mark.parametrize("B,H,Sq,Sk,D,causal,kv_len", [
    (1, 16, 129, 255, 264, False, None), (2, 4, 300, 300, 384, True, None), (1, 8, 384, 384, 512, False, None), (2, 8, 200, 333, 320, False, [333, 129]),
    (2, 8, 200, 333, 392, True, [0, 300]), (1, 1, 500, 2100, 512, False, None), (1, 2, 300, 2049, 328, False, [1030]), (1, 1, 2050, 2050, 456, True, None)])
def test_against_the_oracle(oracle, B, H, Sq, Sk, D, causal, kv_len):
    from flame_amd import capi
    print(f"[two products] {B=} {H=} {Sq=} {Sk=} {D=} {causal=} {kv_len=}", flush=True)
    need, one_pass = _scratch(B, H, Sq, Sk, D)
    assert need >= max(2 * B * H * Sq * Sk, one_pass)
    t = _inputs(8100 + D + Sq, B, H, Sq, Sk, D)
    sc = 1.5 / math.sqrt(D)
    kvl = None if kv_len is None else (kv_len if len(kv_len) == B else kv_len * B)
    ro, rlse, ro32 = oracle.sdpa_fwd(t[0], t[1], t[2], sc, causal=causal, kv_len=kvl, want_f32=True)
    q, k, v = (to_dev(x) for x in t)
    dl = None
    if kvl is not None:
        dl = torch.tensor(kvl, dtype=torch.int32, device="cuda")
        for b, n in enumerate(kvl):                    # what nobody attends to must not be able to reach the output
            k[b, :, n:], v[b, :, n:] = float("nan"), float("nan")
    o = torch.full_like(q, float("nan"))
    _, lse = capi.attn_fwd(q, k, v, sc, causal=causal, kv_len=dl, out=o)
    torch.cuda.synchronize()
    assert_close_bf16(oracle, "O", to_f32(o), ro, ro32)
    glse, fin = lse.cpu().numpy().reshape(rlse.shape), np.isfinite(rlse)
    assert np.array_equal(np.isfinite(glse), fin) and oracle.max_abs(glse[fin], rlse[fin]) <= TOL_LSE


def test_several_launches_and_a_workspace_too_small():
    """16 slices of 2048 x 2048 do not fit the 128 MiB that one launch takes; half the room means the one-pass kernel."""
    from flame_amd import capi
    B, H, S, D = 2, 8, 2048, 392
    need, one_pass = _scratch(B, H, S, S, D)
    assert 2 * 8 * S * S <= need < 2 * 16 * S * S
    g = torch.Generator(device="cuda").manual_seed(3)
    q, k, v = (torch.randn((B, H, S, D), device="cuda", generator=g).to(torch.bfloat16) for _ in range(3))
    o, lse = capi.attn_fwd(q, k, v, D ** -0.5)
    small = torch.empty(need // 2, dtype=torch.uint8, device="cuda")
    o1, lse1 = capi.attn_fwd(q, k, v, D ** -0.5, workspace=small)
    for b in range(B):
        x = torch.matmul(q[b].float(), k[b].float().transpose(-1, -2)) * D ** -0.5
        ref = torch.matmul(torch.softmax(x, -1), v[b].float())
        for got, l in ((o, lse), (o1, lse1)):          # P and O are rounded to bf16, 2^-9 each: 1e-2 as everywhere in these tests
            assert float((got[b].float() - ref).norm() / ref.norm()) <= 1e-2
            assert float((l.view(B, H, S)[b] - torch.logsumexp(x, -1)).abs().max()) <= 1e-3
