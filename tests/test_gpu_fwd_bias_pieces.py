"""The additive-bias forward that loads pieces of 16 bytes and passes them through LDS: layouts of the bias beyond a dense
[1 | B, H, Sq, Sk] (row pitches of any length, rows, heads and batches that are broadcast), more batches than one sharing a bias,
partial wavefronts.  Against the same call on a dense copy of the bias (the same kernel on another layout: bit for bit), which
itself is held to the oracle elsewhere, and against an fp32 reference."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,H,Sq,Sk,D,layout", [
    (3, 2, 33, 130, 64, "pitch"), (1, 3, 140, 67, 128, "pitch"), (2, 5, 129, 128, 64, "rows"), (3, 2, 70, 201, 96, "heads"), (4, 1, 257, 64, 64, "batched")])
def test_layouts(B, H, Sq, Sk, D, layout, dtype):
    from flame_amd import capi
    g = torch.Generator(device="cuda").manual_seed(B * Sq + Sk)
    q, k, v = (torch.randn((B, H, n, D), device="cuda", generator=g).to(torch.bfloat16) for n in (Sq, Sk, Sk))
    if layout == "pitch":
        bias = torch.randn((1, H, Sq, Sk + 5), device="cuda", generator=g).to(dtype)[..., 3:3 + Sk]
    elif layout == "rows":
        bias = torch.randn((1, H, 1, Sk), device="cuda", generator=g).to(dtype)
    elif layout == "heads":
        bias = torch.randn((1, 1, Sq, Sk), device="cuda", generator=g).to(dtype)
    else:
        bias = torch.randn((B, H, Sq, Sk), device="cuda", generator=g).to(dtype)
    o, lse = capi.attn_fwd_bias(q, k, v, D ** -0.5, bias)
    dense = bias.expand(B, H, Sq, Sk).contiguous()
    od, lsed = capi.attn_fwd_bias(q, k, v, D ** -0.5, dense)
    assert torch.equal(o, od) and torch.equal(lse, lsed)
    x = torch.matmul(q.float(), k.float().transpose(-1, -2)) * D ** -0.5 + dense.float()
    ref = torch.matmul(torch.softmax(x, -1), v.float())
    # P and O are rounded to bf16 (2^-9 each, relative): 1e-2 as everywhere in these tests
    assert float((o.float() - ref).norm() / ref.norm()) <= 1e-2
    assert float((lse.view(B, H, Sq) - torch.logsumexp(x, -1)).abs().max()) <= 1e-3
