"""Grids of 256-query workgroups whose last round is cut into smaller workgroups in a launch of its own (32-query ones that share
the keys, or 128-query ones), against the CPU oracle: few left over with whole and with ragged query tiles, and more left
over than the key-sharing ones take.  The backward cuts its last round from two rounds on (128-query ones, with two key groups on
long walks), below that it runs 128-query workgroups throughout: the former against an fp32 reference."""
import pytest
import torch

from flame_amd import workloads as W
from tests.gpu_util import TOL_LSE, assert_close_bf16, recorded_launches, to_dev, to_f32

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


@pytest.mark.parametrize("Sq,Sk,D,groups", [(512, 1088, 64, 1), (450, 1088, 128, 1), (512, 2112, 64, 2), (512, 2112, 128, 2), (500, 1100, 96, 1)])
def test_backward_past_two_rounds(Sq, Sk, D, groups):
    """258 slices of two units: 512 in whole rounds, the last four as eight of 128 queries."""
    from flame_amd import capi
    BH = 258
    print(f"[last round, backward] {BH=} {Sq=} {Sk=} {D=}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(Sq + Sk + D)
    q, k, v, do = (torch.randn((1, BH, n, D), device="cuda", generator=g).bfloat16() for n in (Sq, Sk, Sk, Sq))
    sc = D ** -0.5
    o, lse = capi.attn_fwd(q, k, v, sc)
    grads = capi.attn_bwd(q, k, v, o, do, lse, sc)
    for h0 in range(0, BH, 43):
        a, b, c = (t[0, h0:h0 + 43].float().requires_grad_(True) for t in (q, k, v))
        out = torch.softmax((a @ b.transpose(-1, -2)) * sc, -1) @ c
        want = torch.autograd.grad(out, (a, b, c), do[0, h0:h0 + 43].float())
        for name, x, w in zip(("O", "dQ", "dK", "dV"), (o, *grads), (out.detach(), *want)):
            # P and dS rounded to bf16 (2^-9 each) in sums of many, the result rounded to bf16; per head, so that none is left out
            err = (x[0, h0:h0 + 43].float() - w).flatten(1).norm(dim=1) / w.flatten(1).norm(dim=1)
            assert float(err.max()) <= 1e-2, (name, h0, err)
    DP = 64 if D == 64 else 96 if D == 96 else 128
    got = [x[:2] for x in recorded_launches(lambda: capi.attn_bwd(q, k, v, o, do, lse, sc)) if "bwd_dq" in x[0]]
    assert [n for _, n in got] == [512, 8] and got[0][0].startswith(f"bwd_dq_wide_kernel<{DP}>") and got[1][0].startswith(f"bwd_dq_kernel<{DP}, 0, 4, 0, {groups}>"), got
