"""Room that a call is faster with but does not need: where the device has none left (here: past the limit set for the process) the
kernels that do without serve the call, bit for bit as with a workspace too small; and none is asked for by a call that the
fused kernels refuse."""
import pytest
import torch

pytestmark = pytest.mark.gpu
MIB = 1 << 20


class _Limit:
    """No block above `slack` bytes, whatever room earlier tests left within the segments that the process holds, and at most
    `slack` bytes beyond those."""

    def __init__(self, slack):
        self.slack = slack

    def __enter__(self):
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        total = torch.cuda.get_device_properties(0).total_memory
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + self.slack) / total)
        self.held = []
        try:
            while True:
                self.held.append(torch.empty(self.slack + 1, dtype=torch.uint8, device="cuda"))
        except torch.OutOfMemoryError:
            pass

    def __exit__(self, *exc):
        torch.cuda.set_per_process_memory_fraction(1.0)
        self.held = None


def _randn(g, *shape):
    return torch.randn(shape, device="cuda", generator=g).bfloat16()


def _mask(g, *shape):
    """One byte off alignment: the kernels that read it do not load its rows as vectors, so that bits pay at any size."""
    n = 1
    for x in shape:
        n *= x
    return torch.randint(0, 2, (n + 1,), device="cuda", generator=g, dtype=torch.uint8)[1:].view(shape)


def test_masks_by_query():
    from flame_amd import capi
    B, H, S, D = 2, 32, 2048, 64                       # 64 planes of a mask: 64 MiB of words
    g = torch.Generator(device="cuda").manual_seed(1)
    q, k, v, do = (_randn(g, B, H, S, D) for _ in range(4))
    mask = _mask(g, B, H, S, S)
    none = torch.empty(16, dtype=torch.uint8, device="cuda")
    ws = torch.empty(capi.bwd_workspace_bytes(B, H, S, D), dtype=torch.uint8, device="cuda")
    o, lse = capi.attn_fwd(q, k, v, 0.125, mask=mask, workspace=none)
    want = capi.attn_bwd(q, k, v, o, do, lse, 0.125, mask=mask, workspace=ws)
    o1, lse1, grads = torch.empty_like(o), torch.empty_like(lse), tuple(torch.empty_like(t) for t in (q, k, v))
    with _Limit(4 * MIB):
        capi.attn_fwd(q, k, v, 0.125, mask=mask, out=o1, lse_out=lse1)
        torch.cuda.synchronize()
    assert torch.equal(o, o1) and torch.equal(lse, lse1)
    with _Limit(ws.numel() + 8 * MIB):
        capi.attn_bwd(q, k, v, o, do, lse, 0.125, mask=mask, grads=grads)
        torch.cuda.synchronize()
    for a, b in zip(grads, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("slack,split", [(4 * MIB, False), (100 * MIB, True)])
def test_wide_heads(slack, split):
    """Head dim 512: the probabilities (132 MiB) do not fit; the partial outputs of a key split (32 MiB) do, or neither does."""
    from flame_amd import capi
    B, H, S, D = 1, 1, 8192, 512
    part = capi.fwd_workspace_bytes(B, H, S, S, D)
    assert 0 < part < 98 * MIB
    g = torch.Generator(device="cuda").manual_seed(2)
    q, k, v = (_randn(g, B, H, S, D) for _ in range(3))
    o, lse = capi.attn_fwd(q, k, v, D ** -0.5, workspace=torch.empty(part if split else 16, dtype=torch.uint8, device="cuda"))
    o1, lse1 = torch.empty_like(o), torch.empty_like(lse)
    with _Limit(slack):
        capi.attn_fwd(q, k, v, D ** -0.5, out=o1, lse_out=lse1)
        torch.cuda.synchronize()
    assert torch.equal(o, o1) and torch.equal(lse, lse1)


@pytest.mark.parametrize("D", [160, 36])
def test_a_refused_call_asks_for_none(D):
    from flame_amd import capi
    B, H, S = 1, 4, 1024
    g = torch.Generator(device="cuda").manual_seed(3)
    q, k, v = (_randn(g, B, H, S, D) for _ in range(3))
    o, lse = torch.empty_like(q), torch.empty((B * H, S), device="cuda")
    mask = _mask(g, B, H, S, S)
    asked = lambda: torch.cuda.memory_stats()["requested_bytes.all.allocated"]                        # noqa: E731
    grads = tuple(torch.empty_like(t) for t in (q, k, v))
    before = asked()
    with pytest.raises(capi.FlameAttnError):
        capi.attn_fwd(q, k, v, D ** -0.5, mask=mask, out=o, lse_out=lse)
    assert asked() == before
    with pytest.raises(capi.FlameAttnError):
        capi.attn_bwd(q, k, v, o, q, lse, D ** -0.5, mask=mask, grads=grads)
    assert asked() - before <= capi.bwd_workspace_bytes(B, H, S, D)
