"""A keep-mask that differs by query, turned into bits (taken where the caller has room for them: the native host path asks for
it): documents packed into a sequence, random masks, rows and columns without anything attended, masks per batch, per head and
shared, key lengths and the causal flag on top, lengths that are no multiple of a tile, strides of any kind; forward and
backward against the CPU oracle, and O against the kernels that read the mask itself (no workspace)."""
import numpy as np
import pytest
import torch

from flame_amd import workloads as W
from tests.gpu_util import TOL_LSE, TOL_REL_L2, assert_close_bf16, recorded_launches, to_dev, to_f32

pytestmark = pytest.mark.gpu


def _mask(kind, B, H, Sq, Sk, rng):
    mb, mh = (B if "b" in kind else 1), (H if "h" in kind else 1)
    if kind.startswith("docs"):
        cuts = np.sort(rng.random((mb, mh, 3)), -1)
        dq = (np.arange(Sq)[None, None, :, None] / Sq >= cuts[:, :, None, :]).sum(-1)
        dk = (np.arange(Sk)[None, None, :, None] / Sk >= cuts[:, :, None, :]).sum(-1)
        m = dq[..., :, None] == dk[..., None, :]
    elif kind.startswith("rand"):
        m = rng.random((mb, mh, Sq, Sk)) < 0.7
    else:                      # "ones": whole tiles but for one row, one column, one element
        m = np.ones((mb, mh, Sq, Sk), bool)
        m[..., Sq // 3, :] = False
        m[..., :, Sk // 2] = False
        m[..., Sq - 1, 0] = False
    return m


# (at least 36 tiles of 64 x 64, the sequences rounded up to 128, and rows that do not load as vectors: others, see below)
CASES = [("docs_b", 2, 2, 300, 300, 64, False, None), ("docs", 2, 3, 257, 321, 128, False, None), ("rand_bh", 2, 2, 65, 1153, 72, False, None),
         ("rand", 1, 2, 1090, 64, 128, True, None), ("ones_b", 3, 1, 200, 555, 64, False, [555, 0, 100]), ("ones_h", 1, 3, 383, 383, 96, False, None),
         ("docs_h", 2, 2, 333, 333, 40, True, [333, 77]), ("rand_b", 2, 1, 1200, 1, 64, False, None), ("ones", 1, 2, 2, 1153, 128, False, None)]


@pytest.mark.parametrize("kind,B,H,Sq,Sk,D,causal,kv_len", CASES)
def test_against_the_oracle(oracle, kind, B, H, Sq, Sk, D, causal, kv_len):
    from flame_amd import capi
    print(f"[mask bits] {kind=} {B=} {H=} {Sq=} {Sk=} {D=} {causal=} {kv_len=}", flush=True)
    rng = np.random.default_rng(Sq * Sk + D)
    m = _mask(kind, B, H, Sq, Sk, rng)
    t = [W.f32_to_bf16_bits(W.normal_f32(9000 + Sq + Sk, s, B * H * n * D).reshape(B, H, n, D)) for s, n in enumerate((Sq, Sk, Sk, Sq))]
    sc = D ** -0.5
    full = np.ascontiguousarray(np.broadcast_to(m, (B, H, Sq, Sk)).astype(np.uint8))
    ro, rlse, ro32 = oracle.sdpa_fwd(t[0], t[1], t[2], sc, causal=causal, kv_len=kv_len, mask=full, want_f32=True)
    q, k, v, do = (to_dev(x) for x in t)
    dl = None if kv_len is None else torch.tensor(kv_len, dtype=torch.int32, device="cuda")
    dm = torch.from_numpy(m.astype(np.uint8)).cuda()
    if kind.startswith("rand"):                        # rows apart, keys apart
        wide = torch.zeros((*m.shape[:2], Sq, 2 * Sk + 3), dtype=torch.uint8, device="cuda")
        wide[..., 1:2 * Sk + 1:2] = dm
        dm = wide[..., 1:2 * Sk + 1:2]
    o, lse = capi.attn_fwd(q, k, v, sc, causal=causal, kv_len=dl, mask=dm)
    assert_close_bf16(oracle, "O", to_f32(o), ro, ro32)
    glse, fin = to_f32(lse).reshape(rlse.shape), np.isfinite(rlse)
    assert np.array_equal(np.isfinite(glse), fin) and np.abs(glse[fin] - rlse[fin]).max() <= TOL_LSE
    one = torch.empty(16, dtype=torch.uint8, device="cuda")            # no room: the kernels that read the mask
    o1, lse1 = capi.attn_fwd(q, k, v, sc, causal=causal, kv_len=dl, mask=dm, workspace=one)
    # the same products in another order of the tiles: P against another reference maximum, rounded to bf16
    assert float((o.float() - o1.float()).norm()) <= 5e-3 * float(o1.float().norm()) + 1e-6
    got = capi.attn_bwd(q, k, v, to_dev(ro), do, torch.from_numpy(np.ascontiguousarray(rlse)).cuda().reshape(B * H, Sq), sc, causal=causal, kv_len=dl, mask=dm)
    want = oracle.sdpa_bwd(t[0], t[1], t[2], ro, t[3], sc, causal=causal, kv_len=kv_len, mask=full, want_f32=True)
    for name, g, w, w32 in zip(("dQ", "dK", "dV"), got, want[:3], want[3:]):
        assert_close_bf16(oracle, name, to_f32(g), w, w32)


def test_the_pass_over_the_mask_is_timed():
    """The library's kernel times hold the pass that turns the mask into bits: with the forward, and with dQ."""
    from flame_amd import capi
    g = torch.Generator(device="cuda").manual_seed(4)
    q, k, v, do = (torch.randn((1, 2, 1280, 64), device="cuda", generator=g).bfloat16() for _ in range(4))
    mask = torch.randint(0, 2, (1, 1, 1280, 1280), device="cuda", generator=g, dtype=torch.uint8)
    capi.profiling_enable(True)
    o, lse = capi.attn_fwd(q, k, v, 0.125, mask=mask)
    capi.attn_bwd(q, k, v, o, do, lse, 0.125, mask=mask)
    launches = {kind: n for kind, (_, n) in capi.profiling_read().items() if n}
    capi.profiling_enable(False)
    assert launches == {"fwd": 2, "bwd_dq": 2, "bwd_dkdv": 1}


@pytest.mark.parametrize("H,S,per_head,offset,fwd,bwd", [
    (2, 896, False, 0, False, False), (2, 1024, False, 0, False, True), (2, 1280, False, 0, True, True),
    (2, 1280, True, 0, False, True), (1, 1280, True, 0, True, True),        # of one head: read as often as a shared one
    (2, 896, True, 1, True, True), (2, 833, False, 0, True, True)])         # rows that do not load as vectors
def test_which_kernels_serve_a_mask(H, S, per_head, offset, fwd, bwd):
    """Masks whose rows load as vectors stay with the kernels that read them up to a size, and in the forward where each head
    has its own; the call asks for no room then.  O and the gradients against those of the other kernels."""
    from flame_amd import capi
    g = torch.Generator(device="cuda").manual_seed(S)
    q, k, v, do = (torch.randn((1, H, S, 64), device="cuda", generator=g).bfloat16() for _ in range(4))
    planes = H if per_head else 1
    room = torch.randint(0, 2, (planes * S * S + 16,), device="cuda", generator=g, dtype=torch.uint8)
    mask = room[offset:offset + planes * S * S].view(1, planes, S, S)
    o, lse = capi.attn_fwd(q, k, v, 0.125, mask=mask)
    out, rows, grads = torch.empty_like(o), torch.empty_like(lse), tuple(torch.empty_like(t) for t in (q, k, v))
    for call, bits in ((lambda: capi.attn_fwd(q, k, v, 0.125, mask=mask, out=out, lse_out=rows), fwd),
                       (lambda: capi.attn_bwd(q, k, v, o, do, lse, 0.125, mask=mask, grads=grads), bwd)):
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        call()
        asked = torch.cuda.memory_stats()["allocation.all.allocated"] - before
        names = [name for name, *_ in recorded_launches(call)]
        assert any("mask_bits_kernel" in name for name in names) == bits, names
        if call.__code__.co_names[1:2] == ("attn_fwd",):
            assert asked == int(bits)
    s = (q.float() @ k.float().transpose(-1, -2).contiguous() * 0.125).masked_fill(mask == 0, float("-inf"))
    p = torch.softmax(s, -1)
    dp = do.float() @ v.float().transpose(-1, -2).contiguous()
    ds = p * (dp - (do.float() * (p @ v.float())).sum(-1, keepdim=True)) * 0.125
    want = (p @ v.float(), ds @ k.float(), ds.transpose(-1, -2).contiguous() @ q.float(), p.transpose(-1, -2).contiguous() @ do.float())
    for got, w in zip((out, *grads), want):
        assert float((got.float() - w).norm()) <= TOL_REL_L2 * float(w.norm())
