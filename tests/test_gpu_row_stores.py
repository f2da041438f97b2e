"""Output rows written through LDS: nothing beside the rows and columns of the output is touched, whatever part of a
wavefront's 32 rows exists and wherever the head dim ends.  Outputs are views of a buffer with room around every row, filled
with a pattern; the values are compared with those written into contiguous outputs (the same kernels, so bit for bit)."""
import pytest

torch = pytest.importorskip("torch")
from flame_amd import capi  # noqa: E402
from tests.gpu_util import recorded_launches  # noqa: E402

pytestmark = pytest.mark.gpu
PATTERN = -7.5


def _room(B, H, N, D):
    buf = torch.full((B, N + 2, H, D + 16), PATTERN, device="cuda", dtype=torch.bfloat16)
    return buf, buf[:, 1:N + 1, :, 8:8 + D].permute(0, 2, 1, 3)


def _check(buf, view, want):
    assert torch.equal(view, want)
    view.fill_(PATTERN)
    assert bool((buf == PATTERN).all())


# sizes: a few rows (32 queries per workgroup), partial wavefronts of 128-query workgroups, with two key groups, and 256-query
# workgroups (129 or more rows of the last tile exist, so that they are used): of the forward past one round, of forward and dQ
# in one whole round, also causal
@pytest.mark.parametrize("D", [8, 40, 64, 72, 96, 128])
@pytest.mark.parametrize("B,H,Sq,Sk,causal", [(1, 2, 5, 70, False), (2, 40, 129, 65, False), (1, 24, 1055, 1024, True), (2, 70, 481, 128, False),
                                              (2, 64, 481, 1088, False), (2, 64, 481, 1088, True)])
def test_rows_in_room(D, B, H, Sq, Sk, causal):
    g = torch.Generator(device="cuda").manual_seed(D + Sq)
    q, k, v, do = (torch.randn((B, H, n, D), device="cuda", generator=g).to(torch.bfloat16) for n in (Sq, Sk, Sk, Sq))
    scale = D ** -0.5
    o, lse = capi.attn_fwd(q, k, v, scale, causal=causal)
    buf, view = _room(B, H, Sq, D)
    capi.attn_fwd(q, k, v, scale, causal=causal, out=view)
    _check(buf, view, o)
    want = capi.attn_bwd(q, k, v, o, do, lse, scale, causal=causal)
    bufs = [_room(B, H, n, D) for n in (Sq, Sk, Sk)]
    capi.attn_bwd(q, k, v, o, do, lse, scale, causal=causal, grads=tuple(v for _, v in bufs))
    for (b, w), ref in zip(bufs, want):
        _check(b, w, ref)
    if Sk == 1088:
        names = [name for call in (lambda: capi.attn_fwd(q, k, v, scale, causal=causal), lambda: capi.attn_bwd(q, k, v, o, do, lse, scale, causal=causal))
                 for name, _, _ in recorded_launches(call) if name.startswith(("fwd", "bwd_dq"))]
        compiled = 64 if D <= 64 else 96 if D <= 96 else 128
        fwd = f"fwd_wide_kernel<{compiled}>" if not causal else f"fwd_kernel<{compiled}, 0, {4 if D <= 64 else 8}, 0, 1, false>"
        assert names == [fwd, f"bwd_dq_wide_kernel<{compiled}>"], names
