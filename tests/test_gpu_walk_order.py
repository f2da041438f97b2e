"""The order of unequal walks (the second deal of workgroups turned round, Sage causal walks longest first): every query unit is
worked on exactly once for grids of one, two, three and more deals of the compute units, whole and ragged, causal, with key
lengths and key masks; against an fp32 reference."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _reference(q, k, v, do, sc, keep):
    q, k, v = (t.float().requires_grad_(True) for t in (q, k, v))
    s = ((q @ k.transpose(-1, -2).contiguous()) * sc).masked_fill(~keep, float("-inf"))
    p = torch.softmax(s, -1).nan_to_num(0.0)
    o = p @ v
    return (o, *torch.autograd.grad(o, (q, k, v), do.float()))


@pytest.mark.parametrize("B,H,S,D,kind", [(1, 40, 640, 64, "causal"), (2, 32, 1024, 128, "causal"), (1, 56, 1000, 64, "causal"), (1, 80, 1000, 72, "causal"), (2, 80, 900, 64, "causal"),
                                          (1, 41, 640, 64, "causal"), (8, 8, 700, 64, "kv_len"), (4, 16, 1101, 128, "keys"), (6, 16, 900, 96, "keys")])
def test_every_unit_once(B, H, S, D, kind):
    from flame_amd import capi
    print(f"[walk order] {B=} {H=} {S=} {D=} {kind=}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(B * S + D)
    q, k, v, do = (torch.randn((B, H, S, D), device="cuda", generator=g).bfloat16() for _ in range(4))
    lens = torch.randint(0, S + 1, (B,), device="cuda", generator=g, dtype=torch.int32)
    cols = torch.arange(S, device="cuda")
    kw, keep = dict(causal=True), (cols[None, :] <= cols[:, None])[None, None]
    if kind != "causal":
        keep = (cols[None, :] < lens[:, None])[:, None, None]
        kw = dict(kv_len=lens) if kind == "kv_len" else dict(mask=keep.to(torch.uint8).contiguous())
    sc = D ** -0.5
    o, lse = capi.attn_fwd(q, k, v, sc, **kw)
    grads = capi.attn_bwd(q, k, v, o, do, lse, sc, **kw)
    for b in range(B):
        want = _reference(q[b], k[b], v[b], do[b], sc, keep[b % keep.shape[0]])
        for name, a, w in zip(("O", "dQ", "dK", "dV"), (o, *grads), want):
            # P and dS rounded to bf16 (2^-9 each) in sums of many, the result rounded to bf16
            w = w.detach()
            assert float((a[b].float() - w).norm()) <= 1e-2 * float(w.norm()) + 1e-6, (name, b)


@pytest.mark.parametrize("B,H,S,D", [(1, 40, 640, 64), (1, 24, 2048, 128), (1, 7, 300, 96)])
def test_sage_causal(B, H, S, D):
    from flame_amd import capi
    print(f"[walk order] sage {B=} {H=} {S=} {D=}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(S + D)
    q, k, v = (torch.randn((B, H, S, D), device="cuda", generator=g).bfloat16() for _ in range(3))
    z = capi.sage_quant(q, k)
    o = capi.sage_fwd(z, v, D ** -0.5, causal=True)
    cols = torch.arange(S, device="cuda")
    for h in range(H):
        s = (q[0, h].float() @ (k[0, h].float() - k[0, h].float().mean(0)).t().contiguous()) * D ** -0.5
        w = torch.softmax(s.masked_fill(cols[None, :] > cols[:, None], float("-inf")), -1) @ v[0, h].float()
        # int8 codes: half a step of amax / 127 in every q and k, random: the error of a logit is a few hundredths
        assert float((o[0, h].float() - w).norm()) <= 4e-2 * float(w.norm())
