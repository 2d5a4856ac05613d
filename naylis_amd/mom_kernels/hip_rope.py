"""Fused rotary position embedding of the decoder attention (C ABI: naylis_mom_rope).

transformers' ``apply_rotary_pos_emb`` (called by the Llama attention of each
Naylis decoder layer, model.py:279-345) rotates q and k with five elementwise
ops per tensor; ``rope`` does q and k in one library pass each way with the
same roundings (bitwise equal in bf16 and fp32).  ``NaylisAttention`` is the
Llama attention with that rotation and the same parameters; plain causal bf16
attention with heads of 64 runs on the library's kernels
(``hip_attention.causal_attention``), any other on the configured backend.
"""
from __future__ import annotations

import torch
from transformers.integrations.sdpa_attention import sdpa_attention_forward
from transformers.models.llama.modeling_llama import ALL_ATTENTION_FUNCTIONS, LlamaAttention, eager_attention_forward

from .. import _lib, _torch_ext
from .hip_attention import causal_attention, causal_attention_supported
from .hip_linear import shared_input_linear

_DT = {torch.float32: 0, torch.bfloat16: 1}


def _shape_ok(dtype, device, B, S, hd, cos, sin):
    if torch.version.hip is None or device.type != "cuda" or dtype not in _DT or hd not in (32, 64, 128):
        return False
    for t in (cos, sin):
        if t.dtype != dtype or t.device != device or t.dim() != 3 or t.shape[1:] != (S, hd) \
                or t.shape[0] not in (1, B):
            return False
    return True


def rope_supported(q, k, cos, sin):
    """q, k (B, S, H, hd) of one dtype on a ROCm device, hd 32 / 64 / 128,
    cos / sin (1 or B, S, hd) of the same dtype."""
    if q.dim() != 4 or k.shape != q.shape or k.dtype != q.dtype:
        return False
    B, S, _, hd = q.shape
    return _shape_ok(q.dtype, q.device, B, S, hd, cos, sin)


def rope(q, k, cos, sin):
    """(q', k') = rotary embedding of q, k (B, S, H, hd) with cos / sin
    (1 or B, S, hd); raises when ``rope_supported`` is false."""
    if not rope_supported(q, k, cos, sin):
        raise RuntimeError(f"rope: unsupported inputs q {tuple(q.shape)} {q.dtype} on {q.device}, cos "
                           f"{tuple(cos.shape)} {cos.dtype}")
    q, k = _torch_ext.load().rope(q, k, cos.detach(), sin.detach(), _lib.stream_of(q.device))
    return q, k


class NaylisAttention(LlamaAttention):
    """LlamaAttention with the fused rotation (no cache: the decoder trains and
    evaluates full sequences); other cases run transformers' forward."""

    def _plain_causal(self, attention_mask, kwargs):
        """The SDPA call is softmax(q k^T) v over the causal triangle and
        nothing else: no mask, no dropout, no option of its own, transformers'
        "sdpa" entry not replaced and torch's flash backend (the same
        arithmetic) not switched off by the program."""
        return (self.config._attn_implementation == "sdpa" and attention_mask is None and not kwargs
                and ALL_ATTENTION_FUNCTIONS.get_interface("sdpa", None) is sdpa_attention_forward
                and self.is_causal and self.scaling > 0 and not (self.training and self.attention_dropout)
                and torch.backends.cuda.flash_sdp_enabled())

    def forward(self, hidden_states, position_embeddings=None, attention_mask=None, past_key_values=None,
                **kwargs):
        B, S, _ = hidden_states.shape
        shape = (B, S, -1, self.head_dim)
        cos, sin = position_embeddings
        same_heads = self.q_proj.out_features == self.k_proj.out_features
        dtype = torch.promote_types(hidden_states.dtype, self.q_proj.weight.dtype)
        if past_key_values is not None or not same_heads or \
                not _shape_ok(dtype, hidden_states.device, B, S, self.head_dim, cos, sin):
            return super().forward(hidden_states, position_embeddings=position_embeddings,
                                   attention_mask=attention_mask, past_key_values=past_key_values, **kwargs)
        q, k, v = shared_input_linear(hidden_states, (self.q_proj, self.k_proj, self.v_proj))
        q, k, v = q.view(shape), k.view(shape), v.view(shape)
        q, k = rope(q, k, cos, sin)
        if self._plain_causal(attention_mask, kwargs) and causal_attention_supported(q, k, v):
            return self.o_proj(causal_attention(q, k, v, self.scaling).view(B, S, -1)), None
        interface = ALL_ATTENTION_FUNCTIONS.get_interface(self.config._attn_implementation, eager_attention_forward)
        out, weights = interface(self, q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2), attention_mask,
                                 dropout=0.0 if not self.training else self.attention_dropout, scaling=self.scaling,
                                 **kwargs)
        return self.o_proj(out.reshape(B, S, -1).contiguous()), weights
