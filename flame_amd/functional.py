"""Python-level counterparts of the reference's PyO3 functions for this path
(src/python/functional.rs:187-241 `sdpa`, src/python/nn.rs:390-428 `scaled_dot_product_attention`),
on torch tensors that live on the GPU.  Both are differentiable: the forward saves O and the per-row
log-sum-exp only, the backward recomputes the probabilities tile by tile in the HIP kernels.  The autograd node and
the dispatch between the fused kernels and the materialised path (src/sdpa.rs:483-587 of the reference) are native
(csrc/torch_host.cpp).

Nothing here falls back to torch arithmetic: without the HIP library the calls raise.
"""
from __future__ import annotations

from . import capi


def sdpa(q, k, v, attn_mask=None, is_causal=None, scale=None):
    """Scaled dot-product attention on [B,H,S,D] tensors.

    attn_mask: optional binary keep-mask broadcastable as [B|1, H|1, Sq, Sk] (values >= 0.5 attend; the
    reference's public mask convention, src/sdpa.rs:458-470).  Its buffer may be refilled before the backward: the
    recorded graph holds a copy.  With is_causal=True the mask argument is ignored, as in the reference, and the
    causal structure is applied natively (no mask tensor is built).
    Inputs of another dtype are promoted to bf16 and the result is cast back."""
    return capi.host().sdpa(q, k, v, attn_mask, is_causal is not None and bool(is_causal), scale)


def scaled_dot_product_attention(q, k, v, is_causal=None):
    """nn.scaled_dot_product_attention of the reference: bf16 [B,H,S,D], scale 1/sqrt(D), optional causal."""
    if q.dim() != 4:
        raise ValueError("SDPA expects 4-D input [B, H, S, D]")
    return sdpa(q, k, v, None, is_causal)


def sdpa_with_bias(q, k, v, bias=None, scale=None):
    """attention::sdpa_with_bias: softmax(scale * Q K^T + bias) V with an additive float bias (inference only)."""
    if bias is None:
        return sdpa(q, k, v, scale=scale)
    return capi.host().sdpa_with_bias(q, k, v, bias, scale)
