"""Causal attention of the decoder (C ABI: naylis_mom_attn_*).

The Llama attention inside each Naylis decoder layer (model.py:279-345) reads
its own sequence causally through torch's scaled_dot_product_attention.
``causal_attention`` is that read for bf16 heads of 64 on the library's
kernels, on the projections' (B, S, H, 64) layout both ways.
"""
from __future__ import annotations

import torch

from .. import _lib


def causal_attention_supported(q, k, v):
    """bf16 q, k, v (B, S, H, 64) of one shape on a ROCm device, each sequence
    under 2^31 bytes (512 rows spared, the reach of a tile past its end)."""
    if torch.version.hip is None or not q.is_cuda or q.dim() != 4 or q.shape[3] != 64 or q.numel() == 0:
        return False
    B, S, H, _ = q.shape
    return (q.dtype == k.dtype == v.dtype == torch.bfloat16 and k.shape == q.shape and v.shape == q.shape
            and k.device == q.device and v.device == q.device and B * H <= 1 << 20 and (S + 512) * H * 128 < 0x7fffffff
            and (S + 127) // 128 * B * H < 1 << 31)


class CausalAttentionFunction(torch.autograd.Function):

    @staticmethod
    def forward(ctx, q, k, v, scale):
        lib = _lib.load()
        B, S, H, hd = q.shape
        q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
        dev = q.device
        out = torch.empty_like(q)
        lse = torch.empty((B, H, S), device=dev, dtype=torch.float32)
        with _lib.on_device(dev):
            _lib.check(lib.naylis_mom_attn_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
                                               lse.data_ptr(), scale, B, S, H, hd, _lib.stream_of(dev)))
        ctx.save_for_backward(q, k, v, out, lse)
        ctx.scale = scale
        return out

    @staticmethod
    def backward(ctx, dout):
        lib = _lib.load()
        q, k, v, out, lse = ctx.saved_tensors
        B, S, H, hd = q.shape
        dev = q.device
        dout = dout.to(q.dtype).contiguous()
        dq, dk, dv, delta = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v), torch.empty_like(lse)
        with _lib.on_device(dev):
            _lib.check(lib.naylis_mom_attn_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
                                               lse.data_ptr(), dout.data_ptr(), dq.data_ptr(), dk.data_ptr(),
                                               dv.data_ptr(), delta.data_ptr(), ctx.scale, B, S, H, hd,
                                               _lib.stream_of(dev)))
        return dq, dk, dv, None


def causal_attention(q, k, v, scale):
    """softmax(scale q k^T, causal) v for q, k, v (B, S, H, 64); raises when
    ``causal_attention_supported`` is false."""
    if not causal_attention_supported(q, k, v):
        raise RuntimeError(f"causal_attention: needs bf16 (B, S, H, 64) tensors on a ROCm device; got "
                           f"{tuple(q.shape)} {q.dtype} on {q.device}, {tuple(k.shape)}, {tuple(v.shape)}")
    return CausalAttentionFunction.apply(q, k, v, float(scale))
