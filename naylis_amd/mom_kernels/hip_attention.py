"""Causal attention of the decoder (C ABI: naylis_mom_attn_*).

The Llama attention inside each Naylis decoder layer (model.py:279-345) reads
its own sequence causally through torch's scaled_dot_product_attention.
``causal_attention`` is that read for bf16 heads of 64 on the library's
kernels, on the projections' (B, S, H, 64) layout both ways.
"""
from __future__ import annotations

import torch

from .. import _lib, _torch_ext


def causal_attention_supported(q, k, v):
    """bf16 q, k, v (B, S, H, 64) of one shape on a ROCm device, each sequence
    under 2^31 bytes (512 rows spared, the reach of a tile past its end)."""
    if torch.version.hip is None or not q.is_cuda or q.dim() != 4 or q.shape[3] != 64 or q.numel() == 0:
        return False
    B, S, H, _ = q.shape
    return (q.dtype == k.dtype == v.dtype == torch.bfloat16 and k.shape == q.shape and v.shape == q.shape
            and k.device == q.device and v.device == q.device and B * H <= 1 << 20 and (S + 512) * H * 128 < 0x7fffffff
            and (S + 127) // 128 * B * H < 1 << 31)


def causal_attention(q, k, v, scale):
    """softmax(scale q k^T, causal) v for q, k, v (B, S, H, 64); raises when
    ``causal_attention_supported`` is false."""
    if not causal_attention_supported(q, k, v):
        raise RuntimeError(f"causal_attention: needs bf16 (B, S, H, 64) tensors on a ROCm device; got "
                           f"{tuple(q.shape)} {q.dtype} on {q.device}, {tuple(k.shape)}, {tuple(v.shape)}")
    return _torch_ext.load().causal_attention(q, k, v, float(scale), _lib.stream_of(q.device))
