"""Autograd binding of the layer's bias-free q/o projections with the weight
gradient on the library's split-K MFMA GEMM (C ABI: naylis_mom_linear_wgrad).

model.py:239 (`q_proj`) and model.py:251 (`o_proj`) are nn.Linear(d, d,
bias=False); the reference takes their weight gradient from autograd, a
dy^T x reduction over all B*T tokens.  Here the weight gradient is
naylis_mom_linear_wgrad, deterministic (fixed-order reduction over K ranges or
splits).  The forward product and the input gradient run on the library's GEMM
at the sizes where it is ahead (csrc/torch_nodes.cpp: own_fwd, own_dgrad), as
torch GEMMs (hipBLASLt) otherwise.

The decoder trunk's projections (the Llama attention's q/k/v/o and the MLP's
gate/up/down inside every Naylis decoder layer, model.py:279-345) are the same
bias-free nn.Linear; ``NaylisLinear`` / ``use_library_wgrad`` give them this
weight gradient too, in training at token counts that are multiples of 8 (other
counts train on torch's GEMMs and evaluate on the library's).  At the config-3 shapes (16384 tokens) hipBLASLt's
weight-gradient GEMM runs d x d at about 340 TFLOP/s and d x 2816 at about
620, the library's at about 800 and 950.
"""
from __future__ import annotations

import torch
import torch.nn.functional as F
from torch import nn
from torch.autograd import forward_ad
from torch.nn.modules import module as _modules

from .. import _lib, _torch_ext


def library_wgrad(lib, xin, dy, dtype, dev, st):
    """dW = dy^T xin over all rows: the library's weight gradient where the widths
    are multiples of 8 (any row count), else the torch product that autograd
    would use for nn.Linear's (``lib`` and ``dev`` are xin's)."""
    return _torch_ext.load().linear_wgrad(xin, dy, dtype == torch.float32, st)


def _library_ok(x, weight, rows=8):
    """bf16 x and weight on one ROCm device, widths multiples of 8 and the
    token count a multiple of ``rows``."""
    D_out, D_in = weight.shape
    return (x.is_cuda and torch.version.hip is not None and x.dtype == torch.bfloat16
            and weight.dtype == torch.bfloat16 and weight.device == x.device and D_in > 0 and D_in % 8 == 0
            and D_out % 8 == 0 and x.shape[-1] == D_in and (x.numel() // D_in) % rows == 0)


def _untransformed(x, *weights):
    """Plain tensors outside functorch transforms, forward-mode AD and tracing:
    what may go to a kernel by its pointer where torch's own product, which
    knows about those, ran before."""
    return (type(x) is torch.Tensor and all(type(w) in (torch.Tensor, nn.Parameter) for w in weights)
            and not torch._C._are_functorch_transforms_active() and forward_ad._current_level < 0
            and torch._C._get_tracing_state() is None)


def _plain_module(m):
    """A NaylisLinear whose call is its forward and nothing else: no hooks, its
    own or for all modules, and no forward put on the instance."""
    return (type(m) is NaylisLinear and "forward" not in m.__dict__ and not m._forward_hooks
            and not m._forward_pre_hooks and not _modules._global_forward_hooks
            and not _modules._global_forward_pre_hooks)


def mom_linear(x, weight):
    """y = x W^T (no bias).  For bf16 activations and weights on a ROCm device
    with widths, and in training a token count, that are multiples of 8 the
    weight gradient runs on the library's GEMM, and so do the forward and the
    input gradient at the sizes where it is faster; any other combination is
    the plain torch linear."""
    if not torch.is_grad_enabled():
        if _untransformed(x, weight) and _library_ok(x, weight, 1):
            return _torch_ext.load().linear(x, [weight], False, _lib.stream_of(x.device))[0]
    elif weight.requires_grad and _library_ok(x, weight):
        return _torch_ext.load().shared_linear(x, [weight], _lib.stream_of(x.device))[0]
    return F.linear(x, weight)


def shared_input_linear(x, linears):
    """The outputs of several bias-free linear layers applied to one input,
    as a tuple.  One autograd node for up to three of them (the attention's
    q/k/v, the MLP's gate/up) for bf16 activations and weights on a ROCm device
    with widths and a token count that are multiples of 8: autograd would sum their input
    gradients with separate elementwise adds, the node accumulates each
    further product into the first in the GEMM's epilogue (one rounding of the
    sum).  Where the library's GEMM is faster it takes all forward products in
    one launch, in evaluation too.  Otherwise each layer applied in turn."""
    if len(linears) <= 3 and all(m.bias is None for m in linears):
        ws = [m.weight for m in linears]
        if not torch.is_grad_enabled():
            if _untransformed(x, *ws) and all(_plain_module(m) and _library_ok(x, w, 1)
                                              for m, w in zip(linears, ws)):
                return tuple(_torch_ext.load().linear(x, ws, False, _lib.stream_of(x.device)))
        elif all(_library_ok(x, w) for w in ws) and any(w.requires_grad for w in ws):
            return tuple(_torch_ext.load().shared_linear(x, ws, _lib.stream_of(x.device)))
    return tuple(m(x) for m in linears)


class NaylisLinear(nn.Linear):
    """nn.Linear (same parameters and state-dict keys) whose bias-free form
    runs through ``mom_linear``; with a bias it is nn.Linear's forward."""

    def forward(self, x):
        if self.bias is not None:
            return super().forward(x)
        return mom_linear(x, self.weight)


def use_library_wgrad(module):
    """Turn every bias-free nn.Linear inside ``module`` into a NaylisLinear in
    place (its parameters are untouched).  Returns ``module``."""
    for m in module.modules():
        if type(m) is nn.Linear and m.bias is None:
            m.__class__ = NaylisLinear
    return module
