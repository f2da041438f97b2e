"""A keep-mask of keys (the same for every query): the forward and dQ walk a list of attended 64-key tiles, dK/dV treats it
as a key length with holes.  Against the CPU oracle, forward and backward, at the sizes where the list can go wrong: fewer
keys than a tile, one short of a tile and one past it, tiles without an attended key in front, between and at the end, a
sequence with nothing attended, masks per head, a mask read through a key stride, more tiles than a wavefront has lanes."""
import numpy as np
import pytest
import torch

from flame_amd import workloads as W
from tests.gpu_util import TOL_LSE, assert_close_bf16, to_dev, to_f32

pytestmark = pytest.mark.gpu


def _mask(kind, B, H, Sk, g):
    m = np.ones((B, H, 1, Sk), np.uint8)
    if kind == "lengths":
        for b in range(B):
            m[b, :, :, max(1, Sk * (b + 1) // (B + 1)):] = 0
    elif kind == "holes":
        m[:, :, :, :Sk // 3] = 0
        m[:, :, :, Sk // 2:Sk // 2 + 150] = 0
        m[:, :, :, -3:] = 0
        m[..., Sk // 2 - 1] = 1
    elif kind == "random":
        m[:] = (g.random((B, H, 1, Sk)) < 0.6)
        m[..., 0] = 1
    elif kind == "empty":
        m[0] = 0
    return m


@pytest.mark.parametrize("B,H,Sq,Sk,D,kind,per_head,stride", [
    (2, 2, 70, 33, 64, "lengths", False, 1), (2, 2, 65, 63, 128, "random", True, 1), (1, 3, 128, 64, 64, "ones", False, 1),
    (3, 1, 40, 65, 72, "empty", False, 1), (2, 2, 150, 500, 128, "holes", False, 1), (2, 1, 129, 640, 64, "lengths", True, 2),
    (1, 2, 64, 1101, 128, "holes", True, 1), (1, 1, 33, 4500, 64, "holes", False, 1), (2, 2, 1, 300, 64, "random", False, 1)])
def test_forward_and_backward_against_the_oracle(oracle, B, H, Sq, Sk, D, kind, per_head, stride):
    from flame_amd import capi
    print(f"[key masks] {B=} {H=} {Sq=} {Sk=} {D=} {kind=} {per_head=} {stride=}", flush=True)
    m = _mask(kind, B, H if per_head else 1, Sk, np.random.default_rng(Sk))
    q, k, v, do = (W.f32_to_bf16_bits(W.normal_f32(7500 + Sk, s, B * H * n * D).reshape(B, H, n, D)) for s, n in enumerate((Sq, Sk, Sk, Sq)))
    sc = D ** -0.5
    full = np.ascontiguousarray(np.broadcast_to(m, (B, H, Sq, Sk)))
    ro, rlse, ro32 = oracle.sdpa_fwd(q, k, v, sc, mask=full, want_f32=True)
    rg = oracle.sdpa_bwd(q, k, v, ro, do, sc, mask=full, want_f32=True)
    wide = torch.zeros((*m.shape[:3], Sk * stride), dtype=torch.uint8, device="cuda")
    wide[..., ::stride] = torch.from_numpy(m).cuda()
    mask = wide[..., ::stride]
    dq_, dk_, dv_, do_ = (to_dev(t) for t in (q, k, v, do))
    o, lse = capi.attn_fwd(dq_, dk_, dv_, sc, mask=mask)
    grads = capi.attn_bwd(dq_, dk_, dv_, o, do_, lse, sc, mask=mask)
    torch.cuda.synchronize()
    assert_close_bf16(oracle, "O", to_f32(o), ro, ro32)
    got, fin = to_f32(lse).reshape(rlse.shape), np.isfinite(rlse)
    assert np.array_equal(fin, np.isfinite(got)) and np.abs(got[fin] - rlse[fin]).max(initial=0.0) <= TOL_LSE
    for name, a, bits, f32 in zip(("dQ", "dK", "dV"), grads, rg[:3], rg[3:]):
        assert_close_bf16(oracle, name, to_f32(a), bits, f32)
