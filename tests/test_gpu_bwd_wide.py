"""The backward for head dims above 128 on kernels of its own, against the CPU oracle: head dims that end inside a contraction
step (136, 152, 168, 264), inside a 128-column output tile (192) and on one (512), more key tiles than a band of eight, one row, one past the 128-row tiles, causal with more
keys than queries and the reverse, key lengths (one of them 0), strided views, and a workspace that holds fewer (batch, head)
slices than there are."""
import numpy as np
import pytest
import torch

from flame_amd import workloads as W
from tests.gpu_util import assert_close_bf16, to_dev, to_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,Sq,Sk,D,causal,lens,small_ws,bnhd", [
    (1, 2, 1, 1, 136, False, None, False, False), (1, 2, 100, 77, 264, False, None, False, True), (1, 1, 129, 257, 512, False, None, False, False),
    (2, 2, 128, 128, 192, True, None, True, False), (1, 1, 300, 150, 136, True, None, False, True), (1, 2, 140, 290, 256, True, None, True, False),
    (3, 1, 65, 200, 264, False, (200, 0, 129), True, False),
    (1, 1, 200, 1300, 152, False, None, False, False), (1, 1, 1290, 260, 168, True, None, False, True)])
def test_against_the_oracle(oracle, B, H, Sq, Sk, D, causal, lens, small_ws, bnhd):
    from flame_amd import capi
    print(f"[bwd wide] {B=} {H=} {Sq=} {Sk=} {D=} {causal=} {lens=} {small_ws=} {bnhd=}", flush=True)
    q, k, v, do = (W.f32_to_bf16_bits(W.normal_f32(7700 + Sk, s, B * H * n * D).reshape(B, H, n, D)) for s, n in enumerate((Sq, Sk, Sk, Sq)))
    sc = D ** -0.5
    kvl = None if lens is None else np.asarray(lens, np.int32)
    ro, rlse = oracle.sdpa_fwd(q, k, v, sc, causal=causal, kv_len=kvl)
    rg = oracle.sdpa_bwd(q, k, v, ro, do, sc, causal=causal, kv_len=kvl, want_f32=True)

    def dev(x):
        t = to_dev(x)
        return t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3) if bnhd else t

    ws = None
    if small_ws:        # rows and one slice of P and dS
        pad = lambda n: -(-n // 128) * 128    # noqa: E731
        ws = torch.empty(2 * -(-B * H * Sq * 4 // 256) * 256 + pad(Sq) * pad(Sk) * 4, dtype=torch.uint8, device="cuda")
    grads = tuple(torch.full_like(dev(x), float("nan")) for x in (q, k, v))
    capi.attn_bwd_materialised(dev(q), dev(k), dev(v), dev(ro), dev(do), torch.from_numpy(np.ascontiguousarray(rlse).reshape(B * H, Sq)).cuda(), sc,
                               causal=causal, kv_len=None if kvl is None else torch.from_numpy(kvl).cuda(), workspace=ws, grads=grads)
    torch.cuda.synchronize()
    for name, a, bits, f32 in zip(("dQ", "dK", "dV"), grads, rg[:3], rg[3:]):
        assert_close_bf16(oracle, name, to_f32(a), bits, f32)
