"""What the Python-level sdpa() refuses before it touches the GPU."""
import pytest
import torch


@pytest.mark.parametrize("which", [0, 1, 2])
@pytest.mark.parametrize("recorded", [False, True])
def test_forward_mode(which, recorded):
    """No input requires a gradient, or all do, and one carries a tangent: there is no forward-mode derivative, and a result
    without a tangent would mean a derivative of zero."""
    import torch.autograd.forward_ad as fwad
    from flame_amd import functional as F
    args = [torch.randn(1, 2, 8, 64).to(torch.bfloat16).requires_grad_(recorded) for _ in range(3)]
    with fwad.dual_level():
        args[which] = fwad.make_dual(args[which], torch.ones_like(args[which]))
        for call in (lambda: F.sdpa(*args), lambda: F.scaled_dot_product_attention(*args, is_causal=True), lambda: F.sdpa_with_bias(*args)):
            with pytest.raises(NotImplementedError, match="forward-mode"):
                call()
            with torch.no_grad(), pytest.raises(NotImplementedError, match="forward-mode"):
                call()


@pytest.mark.parametrize("recorded", [False, True])
def test_jit_trace(recorded):
    """The trace would hold the result for its example inputs as a constant."""
    from flame_amd import capi, functional as F
    args = [torch.randn(1, 2, 8, 64).to(torch.bfloat16).requires_grad_(recorded) for _ in range(3)]
    for call in (lambda q, k, v: F.sdpa(q, k, v) * 2, lambda q, k, v: capi.attn_fwd(q, k, v, 0.125)[0] * 2):
        with pytest.raises(RuntimeError, match="cannot be recorded"):
            torch.jit.trace(call, args)
