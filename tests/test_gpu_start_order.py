"""Problems whose slices do not divide by the eight XCDs, more units than compute units: the units left over are dealt one by one
(csrc/causal_order.hpp, csrc/xcd_order.hpp), every one of them once.  Forward and backward against an fp32 reference, head by head."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,Sq,Sk,D,causal,lens,masked", [
    (1, 37, 1024, 1024, 64, True, None, False), (3, 25, 512, 512, 128, True, None, False), (1, 75, 520, 700, 72, True, None, False),
    (9, 12, 300, 400, 64, False, (400, 65, 0, 77, 399, 128, 129, 250, 64), False), (9, 12, 300, 400, 128, False, (50, 400, 300, 77, 20, 128, 129, 250, 64), True),
    (5, 14, 1000, 500, 96, False, (500, 33, 64, 450, 128), False), (1, 43, 850, 200, 128, False, None, False)])
def test_every_unit(B, H, Sq, Sk, D, causal, lens, masked):
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
    o, lse = capi.attn_fwd(q, k, v, sc, **kw)
    grads = capi.attn_bwd(q, k, v, o, do, lse, sc, **kw)
    attend = keep.expand(B, 1, Sq, Sk)
    if causal:
        attend = attend & (torch.arange(Sk, device="cuda")[None] <= torch.arange(Sq, device="cuda")[:, None])
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
