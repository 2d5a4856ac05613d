"""Fused RMSNorm of the Naylis decoder (C ABI: naylis_mom_rmsnorm_*).

The reference builds every norm of its decoder layer — the MoM layer's
pre-norm ``mom_norm`` and the Llama block's two norms — as LlamaRMSNorm, or
as Liger's fused RMSNorm with ``use_liger`` (model.py:304-305):
``h = fp32(x) * rsqrt(mean(fp32(x)^2) + eps); y = weight * h.to(x.dtype)``.
``NaylisRMSNorm`` keeps that module's parameter (``weight``) and ``eps`` and
runs forward and backward as one library pass each.
"""
from __future__ import annotations

import torch
import torch.nn as nn

from .. import _lib, _torch_ext

_DT = {torch.float32: 0, torch.bfloat16: 1}


def rmsnorm_supported(x, weight):
    """True when the fused kernels apply: same-dtype bf16 / fp32 x and weight on
    a ROCm device, D a multiple of 512 in [512, 4096]."""
    D = x.shape[-1]
    return (torch.version.hip is not None and x.is_cuda and x.dtype in _DT and weight.dtype == x.dtype
            and weight.device == x.device and D % 512 == 0 and 512 <= D <= 4096 and weight.shape == (D,))


def rms_norm(x, weight, eps=1e-6):
    """Fused RMSNorm; raises when ``rmsnorm_supported`` is false."""
    if not rmsnorm_supported(x, weight):
        raise RuntimeError(f"rms_norm: needs bf16 / fp32 x and weight of one dtype on a ROCm device with D a "
                           f"multiple of 512 in [512, 4096]; got x {tuple(x.shape)} {x.dtype} on {x.device}, "
                           f"weight {weight.dtype}")
    return _torch_ext.load().rms_norm(x, weight, float(eps), _lib.stream_of(x.device))


class NaylisRMSNorm(nn.Module):
    """Drop-in for LlamaRMSNorm (same ``weight`` parameter and ``eps``,
    ``variance_epsilon`` kept as an alias), computed by the fused kernels."""

    def __init__(self, hidden_size, eps=1e-6):
        super().__init__()
        self.weight = nn.Parameter(torch.ones(hidden_size))
        self.variance_epsilon = eps

    def forward(self, x):
        return rms_norm(x, self.weight, self.variance_epsilon)

    def extra_repr(self):
        return f"{tuple(self.weight.shape)}, eps={self.variance_epsilon}"


def add_rms_norm(x, a, norm):
    """Residual add followed by ``norm``: returns (s, norm(s)) with
    s = x + a.to(x.dtype).  One fused pass when ``norm`` is a NaylisRMSNorm and
    the kernels apply (a in x's dtype or fp32), else the two torch steps."""
    if (isinstance(norm, NaylisRMSNorm) and rmsnorm_supported(x, norm.weight) and a.shape == x.shape
            and a.device == x.device and (a.dtype == x.dtype or a.dtype == torch.float32)):
        s, y = _torch_ext.load().add_rms_norm(x, a, norm.weight, float(norm.variance_epsilon),
                                              _lib.stream_of(x.device))
        return s, y
    s = x + a.to(x.dtype)
    return s, norm(s)
