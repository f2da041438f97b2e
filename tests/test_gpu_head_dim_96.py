"""Head dims 72 to 96 on the kernels compiled for 96: bit for bit what the kernels of 128 give for the same tensors padded with
zeros (the contraction gains zeros only, nothing changes its order), in each of the forms that forward and backward take:
256-query workgroups with and without the causal flag, 128-query ones, key groups, shared walks, split last rounds, key masks,
masks by query, key lengths, dropout."""
import pytest
import torch

from tests.gpu_util import recorded_launches

pytestmark = pytest.mark.gpu
SEED = 0x2545F4914F6CDD1D
# B, H, Sq, Sk, D, causal, kv_len, mask, dropout
CASES = [(2, 32, 1024, 320, 96, False, None, None, 0.0),       # 256-query workgroups, nothing excluded
         (2, 32, 1030, 64, 80, False, None, None, 0.0),        # 128-query ones, ragged
         (2, 36, 1024, 1024, 72, True, None, None, 0.0),       # ... where 256-query ones would have a thin last round, causal
         (2, 20, 500, 333, 96, False, None, None, 0.0), (2, 20, 200, 1, 88, True, None, None, 0.0),
         (1, 24, 900, 2200, 96, False, None, None, 0.0),       # key groups
         (3, 20, 300, 517, 72, False, [517, 0, 65], None, 0.0), (2, 20, 300, 517, 96, False, None, "keys", 0.0),
         (2, 20, 400, 517, 80, True, None, "rows", 0.0), (2, 20, 400, 384, 96, False, None, None, 0.1), (2, 20, 400, 389, 72, True, None, None, 0.1)]


def make(B, H, Sq, Sk, D, kv_len, mask):
    g = torch.Generator(device="cuda").manual_seed(Sq * 7 + Sk + D)
    q, k, v, do = (torch.randn((B, H, n, D), device="cuda", generator=g).bfloat16() for n in (Sq, Sk, Sk, Sq))
    dl = None if kv_len is None else torch.tensor(kv_len, dtype=torch.int32, device="cuda")
    m = None
    if mask is not None:
        m = (torch.rand((B, 1, 1 if mask == "keys" else Sq, Sk), device="cuda", generator=g) < 0.7).to(torch.uint8)
    return q, k, v, do, dl, m


def pad(t):
    return torch.nn.functional.pad(t, (0, 128 - t.shape[-1]))


def same(name, a, b):
    a = a.contiguous().view(torch.int32 if a.dtype == torch.float32 else torch.int16)
    b = b.contiguous().view(torch.int32 if b.dtype == torch.float32 else torch.int16)
    assert torch.equal(a, b), (name, int((a != b).sum()))


def forward(capi, q, k, v, scale, causal, dl, m, p):
    if p:
        return capi.attn_fwd_dropout(q, k, v, scale, p, SEED, causal=causal, kv_len=dl, mask=m)
    return capi.attn_fwd(q, k, v, scale, causal=causal, kv_len=dl, mask=m)


@pytest.mark.parametrize("B,H,Sq,Sk,D,causal,kv_len,mask,p", CASES)
def test_forward_as_padded_to_128(B, H, Sq, Sk, D, causal, kv_len, mask, p):
    from flame_amd import capi
    print(f"[head dim 96] forward {B=} {H=} {Sq=} {Sk=} {D=} {causal=} {kv_len=} {mask=} {p=}", flush=True)
    q, k, v, _, dl, m = make(B, H, Sq, Sk, D, kv_len, mask)
    o, lse = forward(capi, q, k, v, D ** -0.5, causal, dl, m, p)
    o1, lse1 = forward(capi, pad(q), pad(k), pad(v), D ** -0.5, causal, dl, m, p)
    same("O", o, o1[..., :D])
    same("LSE", lse, lse1)


@pytest.mark.parametrize("B,H,Sq,Sk,D,causal,kv_len,mask,p", CASES + [
    (1, 2, 1200, 1200, 80, False, None, None, 0.0),        # shared walks
    (1, 30, 1100, 1100, 72, False, None, None, 0.0),       # the last round of the key blocks split
    (1, 2, 1100, 1100, 96, False, None, None, 0.1)])
def test_backward_as_padded_to_128(B, H, Sq, Sk, D, causal, kv_len, mask, p):
    from flame_amd import capi
    print(f"[head dim 96] backward {B=} {H=} {Sq=} {Sk=} {D=} {causal=} {kv_len=} {mask=} {p=}", flush=True)
    q, k, v, do, dl, m = make(B, H, Sq, Sk, D, kv_len, mask)
    sc = D ** -0.5
    o, lse = forward(capi, q, k, v, sc, causal, dl, m, p)
    f = (lambda *t: capi.attn_bwd_dropout(*t, sc, p, SEED, causal=causal, kv_len=dl, mask=m)) if p else \
        (lambda *t: capi.attn_bwd(*t, sc, causal=causal, kv_len=dl, mask=m))
    for name, a, b in zip(("dQ", "dK", "dV"), f(q, k, v, o, do, lse), f(*(pad(t) for t in (q, k, v, o, do)), lse)):
        same(name, a, b[..., :D])


# The forms of 256-query workgroups: what forward and backward launch (template arguments behind the name, workgroups)
WIDE = [((2, 32, 1024, 1088, 72, True, None, None, 0.0), [("fwd_kernel<96, 0, 8,", 256)], [("bwd_dq_wide_kernel<96>", 256)]),
        ((2, 32, 1024, 1101, 80, False, None, None, 0.0), [("fwd_kernel<96, 0, 8,", 256)], [("bwd_dq_wide_kernel<96>", 256)]),
        ((4, 32, 1024, 1101, 88, False, [1101, 0, 65, 700], None, 0.0), [("fwd_kernel<96, 0, 8,", 512)], [("bwd_dq_wide_kernel<96>", 512)]),
        # a last round in 32-query workgroups, in 128-query ones; of dQ in 128-query ones, with two key groups
        ((1, 65, 1024, 320, 96, False, None, None, 0.0), [("fwd_wide_kernel<96>", 256), ("fwd_keyshare_kernel<128,", 32)], [("bwd_dq_kernel<96, 0, 4, 0, 1>", 520)]),
        ((1, 65, 990, 320, 72, False, None, None, 0.0), [("fwd_wide_kernel<96>", 256), ("fwd_kernel<96, 0, 4, 0, 1,", 8)], [("bwd_dq_kernel<96, 0, 4, 0, 1>", 520)]),
        ((1, 129, 1024, 1088, 80, False, None, None, 0.0), [("fwd_wide_kernel<96>", 512), ("fwd_keyshare_kernel<128,", 32)],
         [("bwd_dq_wide_kernel<96>", 512), ("bwd_dq_kernel<96, 0, 4, 0, 1>", 8)]),
        ((1, 129, 1024, 2112, 96, False, None, None, 0.0), [("fwd_wide_kernel<96>", 512), ("fwd_keyshare_kernel<128,", 32)],
         [("bwd_dq_wide_kernel<96>", 512), ("bwd_dq_kernel<96, 0, 4, 0, 2>", 8)])]


@pytest.mark.parametrize("case,fwd,dq", WIDE)
def test_256_query_workgroups(case, fwd, dq):
    from flame_amd import capi
    B, H, Sq, Sk, D, causal, kv_len, mask, p = case
    test_forward_as_padded_to_128(*case)
    test_backward_as_padded_to_128(*case)
    q, k, v, do, dl, m = make(B, H, Sq, Sk, D, kv_len, mask)
    o, lse = forward(capi, q, k, v, D ** -0.5, causal, dl, m, p)

    def launched(call, like):
        return [(name, groups) for name, groups, _ in recorded_launches(call) if like in name]
    got = launched(lambda: forward(capi, q, k, v, D ** -0.5, causal, dl, m, p), "fwd")
    assert [n for n, _ in fwd] == [name[:len(n)] for (n, _), (name, _) in zip(fwd, got)] and [g for _, g in fwd] == [g for _, g in got], got
    got = launched(lambda: capi.attn_bwd(q, k, v, o, do, lse, D ** -0.5, causal=causal, kv_len=dl, mask=m), "bwd_dq")
    assert [n for n, _ in dq] == [name[:len(n)] for (n, _), (name, _) in zip(dq, got)] and [g for _, g in dq] == [g for _, g in got], got
