"""The additive-bias forward that loads its bias in fours, against the CPU oracle: rows that start at any element's address
(odd key counts), the ragged tail (one key, one short of a tile, one past it), whole tiles only, walks of one to six tiles,
both bias types, broadcast and batched biases, -inf entries."""
import numpy as np
import pytest
import torch

from flame_amd import workloads as W
from tests.gpu_util import TOL_LSE, assert_close_bf16, to_dev, to_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,Sq,Sk,D,batched,dtype", [
    (1, 2, 1, 1, 64, False, "f32"), (2, 2, 40, 63, 64, False, "f32"), (1, 3, 130, 64, 128, True, "f32"), (2, 1, 129, 65, 72, False, "f32"),
    (1, 2, 200, 191, 64, False, "bf16"), (1, 2, 70, 256, 128, True, "bf16"), (2, 2, 128, 321, 64, True, "f32"), (1, 1, 257, 383, 96, False, "bf16")])
def test_against_the_oracle(oracle, B, H, Sq, Sk, D, batched, dtype):
    from flame_amd import capi
    print(f"[bias rows] {B=} {H=} {Sq=} {Sk=} {D=} {batched=} {dtype=}", flush=True)
    q, k, v = (W.f32_to_bf16_bits(W.normal_f32(7400 + Sk, s, B * H * n * D).reshape(B, H, n, D)) for s, n in enumerate((Sq, Sk, Sk)))
    nb = B if batched else 1
    bias = torch.from_numpy(W.normal_f32(7400 + Sk, 5, nb * H * Sq * Sk).reshape(nb, H, Sq, Sk).copy())
    bias[..., Sk // 2] = 3.0
    if Sk > 2:
        bias[..., 1] = float("-inf")
    bias = bias if dtype == "f32" else bias.to(torch.bfloat16)
    sc = 0.5 * D ** -0.5
    ro, rlse, ro32 = oracle.sdpa_fwd_bias(q, k, v, sc, bias.float().numpy(), want_f32=True)
    o, lse = capi.attn_fwd_bias(*(to_dev(t) for t in (q, k, v)), sc, bias.cuda())
    torch.cuda.synchronize()
    assert_close_bf16(oracle, "O", to_f32(o), ro, ro32)
    assert np.abs(to_f32(lse).reshape(rlse.shape) - rlse).max() <= TOL_LSE
