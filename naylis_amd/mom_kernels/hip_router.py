"""Autograd binding of the fused prefix-mean router (C ABI: naylis_mom_router_*).

The reference computes the router with eager torch ops and no kernel boundary
(model.py:169-187, 209-220).  ``mom_route`` returns the same tensors in one
fused launch sequence: (router_logits, router_probs, top_idx, top_gates) and,
on request, the fp32 prefix mean h.  Gradients flow to x, router_down.weight
and router_up.weight from top_gates (the LM path through the read),
router_probs (the aux loss) and router_logits.

``mom_router_stats`` computes the load-balance statistics of a routing
(model.py:476-517) in one library pass; its gradient reaches router_probs as
one (E,) row expanded over the tokens, which the router backward reads with
row stride 0 instead of materialising an (N, E) tensor.
"""
from __future__ import annotations

import torch

from .. import _lib, _torch_ext

_DT = {torch.float32: 0, torch.bfloat16: 1}
NOISE_ADDITIVE, NOISE_GUMBEL_UNIFORM = 0, 1


def d_probs_arg(d_probs, E):
    """(tensor kept alive, device pointer, row stride) for the router
    backward's d_probs: an fp32 (..., E) gradient expanded from one row
    (strides 0 except the last) goes in as that row with stride 0; anything
    else as a dense fp32 copy with stride E."""
    if d_probs is None:
        return None, None, E
    if (d_probs.dtype == torch.float32 and d_probs.stride(-1) == 1
            and all(s == 0 for s in d_probs.stride()[:-1])):
        return d_probs, d_probs.data_ptr(), 0
    dense = d_probs.float().contiguous()
    return dense, dense.data_ptr(), E


def mom_route(x, w_down, w_up, top_k, noise=None, noise_scale=1.0, return_h=False, noise_is_uniform=False):
    """Fused causal prefix-mean router.

    x (B, T, D) bf16 or fp32 on a ROCm device; w_down (R, D), w_up (E, R)
    (cast to fp32: the router computes in fp32 as with fp32 master weights,
    model.py:181-187); noise (B, T, E) or None — added as
    ``noise_scale * noise`` to the logits before top-k only (model.py:209-216).
    With ``noise_is_uniform`` the noise tensor is the uniform draw u of
    model.py:210 and the kernel applies g = -log(-log(u + 1e-9) + 1e-9)
    itself.  Returns (router_logits, router_probs, top_idx int32, top_gates[, h]).
    """
    if x.dim() != 3:
        raise RuntimeError(f"mom_route: x must be (B, T, D), got {tuple(x.shape)}")
    if x.dtype not in _DT:
        raise RuntimeError(f"mom_route: x must be fp32 or bf16, got {x.dtype}")
    if x.device.type != "cuda" or torch.version.hip is None:
        raise RuntimeError(f"mom_route: needs a ROCm device tensor, got {x.device}")
    B, T, D = x.shape
    if w_down.dim() != 2 or w_down.shape[1] != D:
        raise RuntimeError(f"mom_route: router_down weight must be (R, {D}), got {tuple(w_down.shape)}")
    R = w_down.shape[0]
    if w_up.dim() != 2 or w_up.shape[1] != R:
        raise RuntimeError(f"mom_route: router_up weight must be (E, {R}), got {tuple(w_up.shape)}")
    E = w_up.shape[0]
    if noise is not None:
        if noise.shape != (B, T, E):
            raise RuntimeError(f"mom_route: noise must be ({B}, {T}, {E}), got {tuple(noise.shape)}")
        noise = noise.detach().float().contiguous()
    x = x.contiguous()
    w_down = w_down.float().contiguous()
    w_up = w_up.float().contiguous()
    return tuple(_torch_ext.load().route(x, w_down, w_up, noise, float(noise_scale), int(top_k), bool(return_h),
                                         NOISE_GUMBEL_UNIFORM if noise_is_uniform else NOISE_ADDITIVE,
                                         _lib.stream_of(x.device)))


def mom_router_stats(probs, top_idx):
    """Load-balance statistics of one routing: probs (..., E) fp32 router
    softmax, top_idx (..., k) int.  Returns a (2E + 3,) fp32 tensor:
    [0:E] mean prob per block, [E:2E] fraction of tokens selecting it, [2E]
    the aux term E * sum(frac * mean_prob) (model.py:500-503), [2E+1] mean
    router entropy, [2E+2] dead-block fraction (model.py:505-507).  Only
    mean_prob and aux carry gradient (frac comes from the selection mask; the
    reference logs entropy and dead fraction detached)."""
    if probs.dtype != torch.float32:
        probs = probs.float()
    if probs.device.type != "cuda" or torch.version.hip is None:
        raise RuntimeError(f"mom_router_stats: needs a ROCm device tensor, got {probs.device}")
    E = probs.shape[-1]
    if top_idx.shape[:-1] != probs.shape[:-1]:
        raise RuntimeError(f"mom_router_stats: top_idx {tuple(top_idx.shape)} does not match probs "
                           f"{tuple(probs.shape)}")
    return _torch_ext.load().router_stats(probs.contiguous(), top_idx.to(torch.int32).contiguous(),
                                          _lib.stream_of(probs.device))
