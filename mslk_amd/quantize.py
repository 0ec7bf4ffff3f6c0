"""Row-wise FP8 quantization behind the reference's Python interface.

`quantize_fp8_row` keeps the signature, the operator name (`triton::quantize_fp8_row`) and the dispatch of the
reference function (mslk/quantize/triton/fp8_quantize.py:319-378): `use_triton=True` selects the arithmetic of its
GPU kernel, `use_triton=False` the bits of its torch emulation (356-378).  `quantize_fp8_per_row`
(`mslk::quantize_fp8_per_row`) always gives the latter.
"""
from __future__ import annotations

from typing import Optional, Tuple

import torch

FP8_DTYPE = torch.float8_e4m3fn  # gfx950 is OCP FP8 (reference: mslk/utils/device.py:135-160)


def _quantize_fp8_row_fake(a, scale_ub=None, zero_start_index_M=None, use_triton=True, output_device=None,
                           align_rows_to=None, eps_opt=1.0 / 512.0):
    # shape function of the reference (fp8_quantize.py:381-407)
    dev = a.device if output_device is None else output_device
    K = a.shape[-1]
    if align_rows_to is not None:
        K = (K + align_rows_to - 1) // align_rows_to * align_rows_to
    return (torch.empty(tuple(a.shape[:-1]) + (K,), dtype=FP8_DTYPE, device=dev),
            torch.empty(a.shape[:-1], dtype=torch.float32, device=dev))


def _quantize_fp8_per_row_fake(input, bs=None, scale_ub=None, output_dtype=None, stochastic_rounding=False):
    return (torch.empty(input.shape, dtype=FP8_DTYPE, device=input.device),
            torch.empty(input.shape[:-1], dtype=torch.float32, device=input.device))


# Schemas and shape functions; the GPU kernels are native (csrc/torch_ops.cpp, loaded by the package when every schema is defined).
# `triton::quantize_fp8_row` is the operator the reference's torch.library.custom_op (fp8_quantize.py:319-328) defines,
# with its schema and defaults, so a traced or compiled caller of torch.ops.triton.quantize_fp8_row lands here.  When the
# reference defined the op first, only its GPU kernel is replaced; the other way round does not work (the reference's
# custom_op would meet an existing definition), so a process that uses both imports the reference's module first.
# `mslk::quantize_fp8_per_row` has no counterpart in the reference tree: it is a convenience operator under the name the
# path is known by (the legacy FBGEMM operator's signature), always with the torch branch's arithmetic.
_library = torch.library.Library("mslk", "FRAGMENT")
_triton_library = torch.library.Library("triton", "FRAGMENT")
SCHEMAS = {
    "triton::quantize_fp8_row": "quantize_fp8_row(Tensor a, Tensor? scale_ub=None, Tensor? zero_start_index_M=None, "
                                "bool use_triton=True, Device? output_device=None, SymInt? align_rows_to=None, "
                                "float? eps_opt=0.001953125) -> (Tensor, Tensor)",
    "mslk::quantize_fp8_per_row": "quantize_fp8_per_row(Tensor input, Tensor? bs=None, Tensor? scale_ub=None, "
                                  "ScalarType? output_dtype=None, bool stochastic_rounding=False) -> (Tensor, Tensor)",
    "mslk::dequantize_fp8_row": "dequantize_fp8_row(Tensor xq, Tensor x_scale) -> Tensor",
}


def _register_quantize() -> None:
    fakes = {
        "quantize_fp8_row": _quantize_fp8_row_fake,
        "quantize_fp8_per_row": _quantize_fp8_per_row_fake,
        "dequantize_fp8_row": lambda xq, x_scale: torch.empty(xq.shape, dtype=torch.bfloat16, device=xq.device),
    }
    for name, schema in SCHEMAS.items():
        namespace, operator = name.split("::")
        library = _triton_library if namespace == "triton" else _library
        if not hasattr(getattr(torch.ops, namespace), operator):
            library.define(schema)
            torch.library.register_fake(name, fakes[operator], lib=library)


_register_quantize()


def quantize_fp8_row(
    a: torch.Tensor,
    scale_ub: Optional[torch.Tensor] = None,
    zero_start_index_M: Optional[torch.Tensor] = None,
    use_triton: bool = True,
    output_device: Optional[torch.device] = None,
    align_rows_to: Optional[int] = None,
    eps_opt: Optional[float] = 1.0 / 512.0,
) -> Tuple[torch.Tensor, torch.Tensor]:
    """Quantize `a` to e4m3fn with one fp32 scale per row (reference signature and dispatch, fp8_quantize.py:319-378).

    Returns (a_fp8 with a's shape [last dim padded to align_rows_to], scale with shape a.shape[:-1]).
    `use_triton=True` (the default, as in the reference) gives the arithmetic of the reference's GPU kernel: amax
    clamped at `eps_opt` (and `scale_ub`), scale = amax / 448, codes = clamp(a / scale, +-448).  `use_triton=False` gives
    the bits of the reference's torch emulation -- the contract this build is checked against bit for bit: amax clamped
    at 1e-12 in the input dtype, inv = (1 / amax) * 448, codes = cast(a * inv) (values beyond 464 become NaN codes,
    which only happens when `scale_ub` cuts the row maximum), scale = 1 / inv; `eps_opt` has no effect there.
    With `zero_start_index_M` (one entry per [N, K] matrix of the input viewed as [B, M, N, K]) the rows
    n >= zero_start_index_M[b, m] are not read and quantize like all-zero rows (fp8_quantize.py:123-129).
    The input must live on a GPU: there is no CPU implementation in this package.
    """
    if not a.is_cuda:
        raise RuntimeError("mslk_amd.quantize_fp8_row: input must be a GPU tensor (no CPU implementation)")
    return torch.ops.triton.quantize_fp8_row(a, scale_ub, zero_start_index_M, use_triton, output_device, align_rows_to,
                                             eps_opt)


def dequantize_fp8_row(xq: torch.Tensor, x_scale: torch.Tensor) -> torch.Tensor:
    """Row-wise dequantization to bf16 along the last axis (reference signature, fp8_quantize.py:1140-1182):
    out = bf16(float(xq) * x_scale[..., None]), the product taken in fp32."""
    if not xq.is_cuda:
        raise RuntimeError("mslk_amd.dequantize_fp8_row: input must be a GPU tensor (no CPU implementation)")
    return torch.ops.mslk.dequantize_fp8_row(xq, x_scale)


def quantize_fp8_per_row(
    input: torch.Tensor,
    bs: Optional[torch.Tensor] = None,
    scale_ub: Optional[torch.Tensor] = None,
    output_dtype: Optional[torch.dtype] = None,
    stochastic_rounding: bool = False,
) -> Tuple[torch.Tensor, torch.Tensor]:
    """Row amax -> scale = amax / 448 -> e4m3fn codes, bit-exact to the reference's torch emulation
    (`quantize_fp8_row(..., use_triton=False)`, fp8_quantize.py:356-378); the legacy operator name of the path (the
    reference's bench still calls it `CudaFP8Rowwise`, bench/quantize/quantize_ops.py:242-251).  `bs` and stochastic
    rounding are not supported."""
    if not input.is_cuda:
        raise RuntimeError("mslk_amd.quantize_fp8_per_row: input must be a GPU tensor (no CPU implementation)")
    return torch.ops.mslk.quantize_fp8_per_row(input, bs, scale_ub, output_dtype, stochastic_rounding)
