"""Problems whose slices do not divide by the eight XCDs, more units than compute units: the units left over are dealt one by one
(csrc/causal_order.hpp, csrc/xcd_order.hpp), every one of them once.  Forward and backward against an fp32 reference, head by head."""
import pytest
import torch

from tests.gpu_util import recorded_launches

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,Sq,Sk,D,causal,lens,masked", [
    (1, 37, 1024, 1024, 64, True, None, False), (3, 25, 512, 512, 128, True, None, False), (1, 75, 520, 700, 72, True, None, False),
    (9, 12, 300, 400, 64, False, (400, 65, 0, 77, 399, 128, 129, 250, 64), False), (9, 12, 300, 400, 128, False, (50, 400, 300, 77, 20, 128, 129, 250, 64), True),
    (5, 14, 1000, 500, 96, False, (500, 33, 64, 450, 128), False), (1, 43, 850, 200, 128, False, None, False)])
def test_every_unit(B, H, Sq, Sk, D, causal, lens, masked):
    check(B, H, Sq, Sk, D, causal, lens, masked)


def check(B, H, Sq, Sk, D, causal, lens, masked, rows=False):
    """masked: the lengths as a keep-mask of keys; rows: a keep-mask that differs by query on top.  Returns the kernels launched and their workgroups."""
    from flame_amd import capi
    print(f"[start order] {B=} {H=} {Sq=} {Sk=} {D=} {causal=} {lens=} {masked=}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(Sq + Sk + D)
    q, k, v, do = (torch.randn((B, H, n, D), device="cuda", generator=g).bfloat16() for n in (Sq, Sk, Sk, Sq))
    sc = D ** -0.5
    n = torch.tensor(lens or [Sk] * B, dtype=torch.int32, device="cuda")
    keep = (torch.arange(Sk, device="cuda")[None] < n[:, None]).view(B, 1, 1, Sk)
    kw = dict(causal=causal)
    if lens and masked:
        kw["mask"] = keep.to(torch.uint8)
    elif lens:
        kw["kv_len"] = n
    if rows:                                    # documents packed into one sequence
        doc = [torch.arange(m, device="cuda") * 3 // m for m in (Sq, Sk)]
        kw["mask"] = (doc[0][:, None] == doc[1][None]).view(1, 1, Sq, Sk).expand(B, 1, Sq, Sk).to(torch.uint8).contiguous()
        keep = keep & kw["mask"].bool()
    o, lse = capi.attn_fwd(q, k, v, sc, **kw)
    grads = capi.attn_bwd(q, k, v, o, do, lse, sc, **kw)
    attend = keep.expand(B, 1, Sq, Sk)
    if causal:
        attend = attend & (torch.arange(Sk, device="cuda")[None] <= torch.arange(Sq, device="cuda")[:, None])
    attend = attend.expand(B, 1, Sq, Sk)
    for b in range(B):
        a, c, w = (t[b].float().requires_grad_(True) for t in (q, k, v))
        s = ((a @ c.transpose(-1, -2).contiguous()) * sc).masked_fill(~attend[b], float("-inf"))
        out = torch.nan_to_num(torch.softmax(s, -1)) @ w if not bool(attend[b].any(-1).all()) else torch.softmax(s, -1) @ w
        if not bool(attend[b].any()):                          # no key at all: zeros
            want = [torch.zeros_like(t[b].float()) for t in (q, q, k, v)]
        else:
            want = [out.detach(), *torch.autograd.grad(out, (a, c, w), do[b].float())]
        for name, x, y in zip(("O", "dQ", "dK", "dV"), (o, *grads), want):
            # P and dS rounded to bf16 (2^-9 each) in sums of many, the result rounded to bf16; per head, so that none is left out
            diff, size = (x[b].float() - y).flatten(1).norm(dim=1), y.flatten(1).norm(dim=1)
            assert bool((diff <= 1e-2 * size).all()), (name, b, (diff / size).max())
    launched = recorded_launches(lambda: capi.attn_fwd(q, k, v, sc, **kw)) + recorded_launches(lambda: capi.attn_bwd(q, k, v, o, do, lse, sc, **kw))
    return [(name, workgroups) for name, workgroups, _ in launched]


# The kernels compiled for that order, each launched by name: 256-query workgroups under the causal flag and with key lengths, key
# masks, masks as bits (with key lengths too, the only ones by which dK/dV is dealt)
@pytest.mark.parametrize("B,H,Sq,Sk,D,causal,lens,masked,rows,names", [
    (1, 49, 2048, 2112, 128, True, None, False, False, ("fwd_dealt_kernel<128, 0, 8>", "bwd_dq_wide_dealt_kernel<128>", "bwd_dkdv_dealt_kernel<128, false>")),
    (1, 195, 512, 1088, 72, True, None, False, False, ("fwd_kernel<96, 0, 8, 0, 1, false>", "bwd_dq_wide_dealt_kernel<96>", "bwd_dkdv_dealt_kernel<96, false>")),
    (5, 33, 1024, 1088, 128, False, (1088, 64, 1000, 700, 129), False, False,
     ("fwd_dealt_kernel<128, 0, 8>", "bwd_dq_wide_dealt_kernel<128>", "bwd_dkdv_dealt_kernel<128, false>")),
    (5, 33, 1024, 1088, 64, False, (1088, 64, 1000, 700, 129), False, False,
     ("fwd_dealt_kernel<64, 0, 4>", "bwd_dq_wide_dealt_kernel<64>", "bwd_dkdv_dealt_kernel<64, false>")),
    (3, 12, 1000, 1000, 96, False, (1000, 64, 700), True, False, ("fwd_dealt_kernel<96, 5, 4>", "bwd_dq_dealt_kernel<96, 5, 4>", "bwd_dkdv_dealt_kernel<96, false>")),
    (3, 12, 1000, 1000, 64, False, None, False, True, ("fwd_dealt_kernel<64, 6, 4>", "bwd_dq_dealt_kernel<64, 6, 4>", "bwd_dkdv_kernel<64, false, false, false, 0, true>")),
    (3, 12, 1000, 1000, 128, False, (1000, 700, 990), False, True, ("fwd_dealt_kernel<128, 6, 4>", "bwd_dq_dealt_kernel<128, 6, 4>", "bwd_dkdv_dealt_kernel<128, true>"))])
def test_kernels(B, H, Sq, Sk, D, causal, lens, masked, rows, names):
    got = check(B, H, Sq, Sk, D, causal, lens, masked, rows)
    assert [x for x, _ in got if x.startswith(("fwd_", "bwd_d"))] == list(names), got


# slices that divide by eight, one workgroup per compute unit at most, no exclusion at all, one sequence: the kernels without it
@pytest.mark.parametrize("B,H,Sq,Sk,D,causal,lens,masked", [(1, 40, 1024, 1024, 64, True, None, False), (4, 16, 300, 400, 128, False, (400, 65, 0, 77), True),
                                                            (1, 12, 1000, 1000, 128, True, None, False), (1, 37, 1024, 300, 64, False, None, False),
                                                            (1, 12, 3000, 400, 64, False, (333,), False), (1, 12, 3000, 3100, 128, False, (3001,), True)])
def test_other_problems(B, H, Sq, Sk, D, causal, lens, masked):
    got = check(B, H, Sq, Sk, D, causal, lens, masked)
    assert not any("dealt" in x for x, _ in got), got


@pytest.mark.parametrize("B,H,S,D,lens", [(1, 37, 1024, 64, None), (1, 37, 1024, 128, None), (3, 12, 1000, 128, (1000, 70, 600)), (5, 12, 640, 64, (640, 70, 600, 64, 333))])
def test_sage(B, H, S, D, lens):
    from flame_amd import capi
    print(f"[start order] sage {B=} {H=} {S=} {D=} {lens=}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(S + D)
    q, k, v = (torch.randn((B, H, S, D), device="cuda", generator=g).bfloat16() for _ in range(3))
    n = torch.tensor(lens or [S] * B, dtype=torch.int32, device="cuda")
    z = capi.sage_quant(q, k)

    def call():
        return capi.sage_fwd(z, v, D ** -0.5, causal=lens is None, kv_len=n if lens else None)
    o = call()
    (name, _, _), = recorded_launches(call)
    assert name == f"sage_fwd_dealt_kernel<{D}, 4>", name
    cols = torch.arange(S, device="cuda")
    sq, sk = (z[x].repeat_interleave(m, 2)[:, :, :S, None] for x, m in (("sq", 128), ("sk", 64)))       # the scales of blocks of rows
    for b in range(B):
        logits = (z["qi8"][b].float() * sq[b]) @ (z["ki8"][b].float() * sk[b]).transpose(-1, -2).contiguous() * D ** -0.5
        gone = cols[None, :] > cols[:, None] if lens is None else (cols >= n[b])[None]
        want = torch.softmax(logits.masked_fill(gone, float("-inf")), -1) @ v[b].float()
        # P rounded to bf16 (2^-9) in sums of many, the result rounded to bf16; per head, so that none is left out
        diff, size = (o[b].float() - want).flatten(1).norm(dim=1), want.flatten(1).norm(dim=1)
        assert bool((diff <= 1e-2 * size).all()), (b, (diff / size).max())
