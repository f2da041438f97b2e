"""Head dims 72 to 96 on the kernels compiled for 96: bit for bit what the kernels of 128 give for the same tensors padded with
zeros (the contraction gains zeros only, nothing changes its order), in each of the forms that forward and backward take:
256-query workgroups with and without the causal flag, 128-query ones, key groups, shared walks, split last rounds, key masks,
masks by query, key lengths, dropout."""
import pytest
import torch

pytestmark = pytest.mark.gpu
SEED = 0x2545F4914F6CDD1D
# B, H, Sq, Sk, D, causal, kv_len, mask, dropout
CASES = [(2, 32, 1024, 320, 96, False, None, None, 0.0),       # 256-query workgroups, nothing excluded
         (2, 32, 1030, 64, 80, False, None, None, 0.0),        # ... with a last round cut off
         (2, 36, 1024, 1024, 72, True, None, None, 0.0),       # 256-query workgroups, causal
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
