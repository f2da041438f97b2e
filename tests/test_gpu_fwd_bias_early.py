"""The bias of D = 64 requested one step ahead: walks of one to eleven tiles that end with a whole or a ragged one (the steps that
copy two whole tiles, those that copy none, an odd pair between them), both bias types, a batch of biases, partial wavefronts;
against an fp32 reference."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("Sk", [64, 100, 128, 192, 200, 256, 320, 321, 384, 449, 512, 640, 703])
def test_walks(Sk, dtype):
    from flame_amd import capi
    print(f"[bias early] {Sk=} {dtype=}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(Sk)
    B, H, Sq, D = 2, 3, 140, 64
    q, k, v = (torch.randn((B, H, n, D), device="cuda", generator=g).bfloat16() for n in (Sq, Sk, Sk))
    bias = (2 * torch.randn((B, H, Sq, Sk), device="cuda", generator=g)).to(dtype)       # a tile's bias taken for another's shows
    o, lse = capi.attn_fwd_bias(q, k, v, 0.125, bias)
    for b in range(B):
        s = 0.125 * (q[b].float() @ k[b].float().transpose(-1, -2).contiguous()) + bias[b].float()
        want = torch.softmax(s, -1) @ v[b].float()
        # P and O rounded to bf16 (2^-9 each)
        assert float((o[b].float() - want).norm()) <= 5e-3 * float(want.norm())
        assert float((lse.view(B, H, Sq)[b] - torch.logsumexp(s, -1)).abs().max()) <= 2e-3
