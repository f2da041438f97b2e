"""fp32 Q, K and V of a call without a graph: bit for bit the call on their bf16 roundings, back in fp32; layouts, views of larger
tensors, expanded heads, odd addresses, infinities and NaN; what the one-launch conversion does not take (a last axis that is not
contiguous, head dims that are no multiple of 8, mixed types, large tensors) gives the same through the tensor library."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _check(q, k, v, **kw):
    from flame_amd import functional as F
    with torch.no_grad():
        got = F.sdpa(q, k, v, **kw)
        want = F.sdpa(*(t.bfloat16().contiguous() for t in (q, k, v)), **kw).to(q.dtype)
    assert got.dtype == q.dtype and got.shape == want.shape
    assert torch.equal(torch.nan_to_num(got, nan=7.0), torch.nan_to_num(want, nan=7.0))


@pytest.mark.parametrize("B,H,Sq,Sk,D", [(1, 1, 2, 3, 8), (2, 12, 77, 77, 64), (1, 5, 130, 257, 80), (3, 2, 64, 33, 128), (1, 2, 40, 70, 512), (2, 3, 50, 60, 36), (1, 33, 1000, 1000, 128)])
@pytest.mark.parametrize("form", ["bhnd", "bnhd", "slice", "expanded", "offset", "last_axis", "mixed"])
def test_as_rounded_first(B, H, Sq, Sk, D, form):
    print(f"[fp32 inputs] {B=} {H=} {Sq=} {Sk=} {D=} {form=}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(Sq + Sk + D)
    rnd = lambda *s: torch.randn(s, device="cuda", generator=g)                     # noqa: E731
    if form == "bnhd":
        q, k, v = (rnd(B, n, H, D).transpose(1, 2) for n in (Sq, Sk, Sk))
    elif form == "slice":                               # of one projection
        x = rnd(B, max(Sq, Sk), 3, H, D)
        q, k, v = (x[:, :n, i].transpose(1, 2) for i, n in enumerate((Sq, Sk, Sk)))
    elif form == "expanded":
        q, k, v = rnd(B, H, Sq, D), rnd(B, 1, Sk, D).expand(B, H, Sk, D), rnd(1, H, Sk, D).expand(B, H, Sk, D)
    elif form == "offset":                              # rows that start on 4 bytes only
        q, k, v = (rnd(B, H, n, D + 3)[..., 3:] for n in (Sq, Sk, Sk))
    elif form == "last_axis":
        q, k, v = (rnd(B, H, D, n).transpose(2, 3) for n in (Sq, Sk, Sk))
    else:
        q, k, v = rnd(B, H, Sq, D), rnd(B, H, Sk, D), rnd(B, H, Sk, D)
    if form == "mixed":
        v = v.bfloat16()
    _check(q, k, v)


def test_special_values_and_graph():
    from flame_amd import functional as F
    g = torch.Generator(device="cuda").manual_seed(5)
    q, k, v = (torch.randn((1, 2, 100, 64), device="cuda", generator=g) for _ in range(3))
    v[0, 0, 3, 5], v[0, 1, 7, 1], q[0, 1, 9, 0], v[0, 0, 50, 2] = float("inf"), float("-inf"), float("nan"), 3.4e38
    _check(q, k, v, is_causal=True)
    mask = torch.rand((1, 1, 100, 100), device="cuda", generator=g) < 0.7
    _check(q, k, v, attn_mask=mask)
    v = torch.randn((1, 2, 100, 64), device="cuda", generator=g)
    a = [t.detach().nan_to_num(0.0).requires_grad_(True) for t in (q, k, v)]        # a graph: recorded as before
    F.sdpa(*a).sum().backward()
    assert all(t.grad is not None and t.grad.dtype == torch.float32 and bool(t.grad.isfinite().all()) for t in a)


def test_a_dispatch_mode_sees_the_conversions():
    """... as they were before the one-launch conversion, which calls outside of such a mode take."""
    from torch.utils._python_dispatch import TorchDispatchMode
    from flame_amd import functional as F
    from tests.gpu_util import recorded_launches

    class Seen(TorchDispatchMode):
        def __init__(self):
            super().__init__()
            self.names = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.names.append(func.name())
            return func(*args, **(kwargs or {}))

    g = torch.Generator(device="cuda").manual_seed(6)
    q, k, v = (torch.randn((1, 2, 100, 64), device="cuda", generator=g) for _ in range(3))
    want = F.sdpa(q, k, v)
    with Seen() as seen:
        got = F.sdpa(q, k, v)
    assert seen.names.count("aten::_to_copy") == 4          # Q, K, V and the output
    assert torch.equal(got, want)
    assert any("cast_qkv_kernel" in name for name, _, _ in recorded_launches(lambda: F.sdpa(q, k, v)))
