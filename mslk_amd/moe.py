"""Fused producers of the FP8 activations of the MoE GEMMs, behind the reference's Python interface.

`silu_mul_quant` (mslk/moe/activation.py:72-135) and `gather_scale_quant_dense_tokens`
(mslk/moe/gather_scatter.py:96-170) keep the reference's signatures and are also registered as
`torch.ops.mslk.silu_mul_quant` / `torch.ops.mslk.gather_scale_quant_dense_tokens` (GPU kernels
only, native: csrc/torch_ops.cpp).  The second op's schema declares the tuple it really returns (the reference's schema string
says `-> Tensor` while its kernels return two tensors).
"""
from __future__ import annotations

from typing import Optional, Tuple

import torch

from .quantize import FP8_DTYPE


def _fake_silu_mul_quant(x0, x1, scale_ub=None, valid_token_count=None):
    return (torch.empty(x0.shape, device=x0.device, dtype=FP8_DTYPE),
            torch.empty((x0.shape[0],), device=x0.device, dtype=torch.float32))


def _fake_gather_scale_quant(x, token_indices, expert_indices, scores, scale_ub=None, valid_token_count=None):
    # mslk/moe/gather_scatter.py:331-345
    a, D = token_indices.shape[0], x.shape[1]
    return (torch.empty((a, D), device=x.device, dtype=FP8_DTYPE), torch.empty((a,), device=x.device, dtype=torch.float32))


_library = torch.library.Library("mslk", "FRAGMENT")
_OPS = {
    "silu_mul_quant": ("(Tensor x0, Tensor x1, Tensor? scale_ub=None, Tensor? valid_token_count=None) -> (Tensor, Tensor)",
                       _fake_silu_mul_quant),
    "gather_scale_quant_dense_tokens": (
        "(Tensor x, Tensor token_indices, Tensor expert_indices, Tensor scores, Tensor? scale_ub=None, "
        "Tensor? valid_token_count=None) -> (Tensor, Tensor)", _fake_gather_scale_quant),
}
for _name, (_schema, _fake) in _OPS.items():
    if not hasattr(torch.ops.mslk, _name):
        _library.define(_name + _schema)
        torch.library.register_fake(f"mslk::{_name}", _fake, lib=_library)


def silu_mul_quant(x0: torch.Tensor, x1: torch.Tensor, scale_ub: Optional[torch.Tensor] = None,
                   valid_token_count: Optional[torch.Tensor] = None) -> Tuple[torch.Tensor, torch.Tensor]:
    """y, y_scale = quantize(x0 * sigmoid(x0) * x1) for x0, x1 of shape (T, D); rows at or beyond
    valid_token_count[0] are left uninitialised (reference signature, mslk/moe/activation.py:72-93)."""
    if not x0.is_cuda:
        raise RuntimeError("mslk_amd.silu_mul_quant: inputs must be GPU tensors (no CPU implementation)")
    return torch.ops.mslk.silu_mul_quant(x0, x1, scale_ub, valid_token_count)


def gather_scale_quant_dense_tokens(x: torch.Tensor, token_indices: torch.Tensor, expert_indices: torch.Tensor,
                                    scores: torch.Tensor, scale_ub: Optional[torch.Tensor] = None,
                                    valid_token_count: Optional[torch.Tensor] = None
                                    ) -> Tuple[torch.Tensor, torch.Tensor]:
    """out[i] = quantize(x[token_indices[i]] * scores[token_indices[i], expert_indices[i]])
    (reference signature, mslk/moe/gather_scatter.py:96-128)."""
    if not x.is_cuda:
        raise RuntimeError("mslk_amd.gather_scale_quant_dense_tokens: inputs must be GPU tensors (no CPU implementation)")
    return torch.ops.mslk.gather_scale_quant_dense_tokens(x, token_indices, expert_indices, scores, scale_ub,
                                                          valid_token_count)
