"""`torch.ops.mslk.*` rowwise FP8 GEMM operators backed by the gfx950 HIP kernels.

The schema strings are the reference's (csrc/gemm/gemm_ops.cpp:31-44,88-96), so callers written
against `torch.ops.mslk.f8f8bf16_rowwise` etc. run unchanged.  When the reference's own library has
already defined a schema, only the GPU ("CUDA" dispatch key) kernel is replaced -- the same seam
the reference's Python kernels use (mslk/gemm/flydsl/preshuffle_gemm.py:433-475).

The kernels of the operators on the hot path are native (csrc/torch_ops.cpp): argument checks, allocation and the call of
the C ABI without the interpreter; the padded-rows and batched forms are the Python functions below.
Validation and error messages follow the reference's ROCm host wrappers
(csrc/gemm/ck/fp8_rowwise/fp8fp8bf16_rowwise_gemm.hip:499-550,
 csrc/gemm/ck/fp8_rowwise_grouped/fp8_rowwise_grouped_gemm.hip:481-559,607-655), except that `bias`
is implemented (semantics of csrc/gemm/cutlass/f8f8bf16_rowwise/f8f8bf16_rowwise_common.cuh:150-198:
per-column fp32 or bf16 bias added after both scales) instead of rejected.
Only GPU kernels are registered: calling these ops with CPU tensors is a dispatcher error.
"""
from __future__ import annotations

from typing import List, Optional, Sequence

import torch

from . import _lib

FP8_DTYPE = torch.float8_e4m3fn

_SCHEMAS = {
    "f8f8bf16_rowwise": "(Tensor XQ, Tensor WQ, Tensor x_scale, Tensor w_scale, Tensor? bias=None, bool use_fast_accum=True) -> Tensor",
    "f8f8bf16_rowwise_out": "(Tensor XQ, Tensor WQ, Tensor x_scale, Tensor w_scale, Tensor(a!) output, Tensor? bias=None, bool use_fast_accum=True) -> ()",
    "f8f8f16_rowwise": "(Tensor XQ, Tensor WQ, Tensor x_scale, Tensor w_scale, Tensor? bias=None, bool use_fast_accum=True) -> Tensor",
    "f8f8bf16_rowwise_preshuffle": "(Tensor XQ, Tensor WQ, Tensor x_scale, Tensor w_scale, Tensor? bias=None, bool use_fast_accum=True) -> Tensor",
    "f8f8f16_rowwise_preshuffle": "(Tensor XQ, Tensor WQ, Tensor x_scale, Tensor w_scale, Tensor? bias=None, bool use_fast_accum=True) -> Tensor",
    "f8f8bf16_rowwise_grouped": "(Tensor[] XQ, Tensor[] WQ, Tensor[] x_scale, Tensor[] w_scale) -> Tensor[]",
    "f8f8bf16_rowwise_grouped_cat": "(Tensor[] XQ, Tensor[] WQ, Tensor[] x_scale, Tensor[] w_scale) -> Tensor",
    "f8f8bf16_rowwise_grouped_stacked": "(Tensor XQ, Tensor WQ, Tensor x_scale, Tensor w_scale, Tensor M_sizes) -> Tensor",
    "f8f8bf16_rowwise_grouped_dynamic": "(Tensor XQ, Tensor WQ, Tensor x_scale, Tensor w_scale, Tensor zero_start_index_M, bool zeroing_output_tensor=True) -> Tensor",
    "f8f8bf16_rowwise_grouped_mm": "(Tensor XQ, Tensor WQ, Tensor x_scale, Tensor w_scale, Tensor? offsets, Tensor(a!) output) -> Tensor",
    "f8f8bf16_rowwise_batched": "(Tensor XQ, Tensor WQ, Tensor x_scale, Tensor w_scale, Tensor? bias=None, bool use_fast_accum=True, Tensor(a!)? output=None) -> Tensor",
    # no counterpart in the reference: its quantize_fp8_row -> f8f8bf16_rowwise pair as one operator (one launch at decode sizes)
    "quantize_f8f8bf16_rowwise": "(Tensor X, Tensor WQ, Tensor w_scale, Tensor? bias=None) -> (Tensor, Tensor, Tensor)",
}

_library = torch.library.Library("mslk", "FRAGMENT")


try:   # the raw handle of the current stream without building a Stream object (4 us -> 0.3 us per call)
    from torch._C import _cuda_getCurrentRawStream as _raw_stream
except ImportError:   # pragma: no cover
    _raw_stream = None


def _stream_ptr(device: torch.device) -> int:
    if _raw_stream is not None:
        return _raw_stream(device.index if device.index is not None else torch.cuda.current_device())
    return torch.cuda.current_stream(device).cuda_stream


class _on_device:
    """`with torch.cuda.device(d)` only when d is not already current (the switch costs microseconds)."""

    __slots__ = ("ctx",)

    def __init__(self, device: torch.device):
        self.ctx = None if device.index in (None, torch.cuda.current_device()) else torch.cuda.device(device)

    def __enter__(self):
        if self.ctx is not None:
            self.ctx.__enter__()

    def __exit__(self, *exc):
        if self.ctx is not None:
            self.ctx.__exit__(*exc)


def _check(cond: bool, msg: str = "") -> None:
    if not cond:
        raise RuntimeError(msg or "Expected condition to be true (mslk_amd argument check)")


def _bias_args(bias: Optional[torch.Tensor], N: int, device: torch.device):
    if bias is None:
        return None, 0, None
    _check(bias.device == device, "bias must be on the same device as XQ")
    _check(bias.dtype in (torch.float32, torch.bfloat16), "Bias type must be bfloat16 or float32 if provided.")
    _check(bias.numel() == N, f"bias must have N={N} elements, got {bias.numel()}")
    b = bias.contiguous()
    return b.data_ptr(), (1 if b.dtype == torch.float32 else 2), b


def _op(name: str, *args):
    """The registered operator, outside of autograd: these products have no derivative, and autograd's fallback for such an
    operator would make its results, and an output it writes, part of the graph of any input that requires a gradient."""
    op = getattr(torch.ops.mslk, name)
    if not torch.is_grad_enabled():
        return op(*args)
    with torch.no_grad():
        return op(*args)


def _rowwise_impl(XQ, WQ, x_scale, w_scale, bias, use_fast_accum, output=None, out_dtype=torch.bfloat16,
                  preshuffled=False):
    if not XQ.is_cuda:   # what the operator's kernel checks in front of this, in its order (without a GPU tensor there is no kernel)
        _check(XQ.dtype == WQ.dtype, f"XQ and WQ dtypes must match, got {XQ.dtype} vs {WQ.dtype}")
        _check(XQ.dtype == FP8_DTYPE, f"XQ and WQ must be {FP8_DTYPE} on gfx950, got {XQ.dtype}")
        _check(x_scale.dtype == torch.float32 and w_scale.dtype == torch.float32, "Scales must be float32.")
        _check(use_fast_accum, "AMD does not support disabling use_fast_accum.")
        _check(False, "XQ must be a contiguous GPU tensor")
    if output is not None:
        _op("f8f8bf16_rowwise_out", XQ, WQ, x_scale, w_scale, output, bias, use_fast_accum)
        return output
    name = ("f8f8f16_rowwise" if out_dtype == torch.float16 else "f8f8bf16_rowwise") + ("_preshuffle" if preshuffled else "")
    return _op(name, XQ, WQ, x_scale, w_scale, bias, use_fast_accum)


def f8f8bf16_rowwise(XQ, WQ, x_scale, w_scale, bias=None, use_fast_accum=True):
    return _rowwise_impl(XQ, WQ, x_scale, w_scale, bias, use_fast_accum)


def f8f8bf16_rowwise_out(XQ, WQ, x_scale, w_scale, output, bias=None, use_fast_accum=True):
    _rowwise_impl(XQ, WQ, x_scale, w_scale, bias, use_fast_accum, output)


def quantize_f8f8bf16_rowwise(X, WQ, w_scale, bias=None):
    """bf16 activations in, bf16 out: `quantize_fp8_row(X, use_triton=False)` followed by `f8f8bf16_rowwise`, returning
    (Y, XQ, x_scale) -- the pair every decode step of a caller of the reference issues (bench/gemm/gemm_ops.py:593-673).
    For 1 <= M <= 4 rows of bf16 with K % 128 == 0 (K >= 1024) it is ONE launch (every workgroup quantizes the rows itself; XQ and
    x_scale are the bits the stand-alone quantizer returns); other shapes run the two kernels."""
    if not X.is_cuda:
        _check(WQ.dtype == FP8_DTYPE, f"WQ must be {FP8_DTYPE} on gfx950, got {WQ.dtype}")
        _check(w_scale.dtype == torch.float32, "Scales must be float32.")
        _check(False, "WQ must be a contiguous 2-D GPU tensor")
    return _op("quantize_f8f8bf16_rowwise", X, WQ, w_scale, bias)


def f8f8f16_rowwise(XQ, WQ, x_scale, w_scale, bias=None, use_fast_accum=True):
    """Same GEMM with an fp16 result (fp8fp8fp16_rowwise_gemm.hip:66-133)."""
    return _rowwise_impl(XQ, WQ, x_scale, w_scale, bias, use_fast_accum, None, torch.float16)


def f8f8bf16_rowwise_preshuffle(XQ, WQ, x_scale, w_scale, bias=None, use_fast_accum=True):
    """f8f8bf16_rowwise on weights pre-shuffled by `ck_preshuffle(wq, 16)` / `preshuffle_b_mfma(wq)`
    (fp8_rowwise_preshuffle_gemm.hip:93-171)."""
    return _rowwise_impl(XQ, WQ, x_scale, w_scale, bias, use_fast_accum, None, torch.bfloat16, True)


def f8f8f16_rowwise_preshuffle(XQ, WQ, x_scale, w_scale, bias=None, use_fast_accum=True):
    """fp16-output variant.  (The reference registers its bf16 function under this name too,
    gemm_ops.cpp:145; the schema and the fp16 wrapper at fp8_rowwise_preshuffle_gemm.hip:160-171 say fp16.)"""
    return _rowwise_impl(XQ, WQ, x_scale, w_scale, bias, use_fast_accum, None, torch.float16, True)


def preshuffle_b_mfma(src: torch.Tensor) -> torch.Tensor:
    """FP8 weights [N, K] or [G, N, K] -> the blocked order [N/16][K/64][4][16][16 B] the *_preshuffle GEMMs
    read (mslk/quantize/shuffle.py:208-246).  Same shape and dtype as `src`; out of place."""
    _check(src.is_cuda and src.is_contiguous(), "preshuffle_b_mfma: src must be a contiguous GPU tensor")
    _check(src.element_size() == 1 and src.dim() in (2, 3), "preshuffle_b_mfma: src must be an 8-bit [N, K] or [G, N, K] tensor")
    N, K = src.shape[-2], src.shape[-1]
    if N % 16 or K % 64:
        raise ValueError(f"preshuffle_b_mfma needs N % 16 == 0 and K % 64 == 0, got N={N} K={K}")
    G = src.shape[0] if src.dim() == 3 else 1
    dst = torch.empty_like(src)
    if src.numel():
        with _on_device(src.device):
            _lib.check(_lib.lib().mslk_amd_preshuffle_b(src.data_ptr(), dst.data_ptr(), G, N, K, _stream_ptr(src.device)))
    return dst


def ck_preshuffle(src: torch.Tensor, NXdl: int = 16) -> torch.Tensor:
    """Reference name for the same re-layout of one [N, K] matrix (mslk/quantize/shuffle.py:182-205);
    only the 16-row wave tile the GEMM reads is supported."""
    _check(NXdl == 16, "ck_preshuffle: only NXdl = 16 is supported")
    _check(src.dim() == 2, "ck_preshuffle: src must be [N, K]")
    return preshuffle_b_mfma(src)


def _check_grouped(XQ: Sequence[torch.Tensor], WQ, x_scale, w_scale) -> None:
    """The argument checks of the TensorList ops in front of their kernel; the kernel makes the others."""
    _check(len(XQ) == len(WQ) == len(x_scale) == len(w_scale), "All inputs must have the same number of groups.")
    if len(XQ) > 0 and not XQ[0].is_cuda:
        _check(XQ[0].dtype == FP8_DTYPE, f"XQ and WQ must be {FP8_DTYPE} on gfx950, got {XQ[0].dtype}")
        _check(False, "XQ tensors must be contiguous GPU tensors")


def f8f8bf16_rowwise_grouped(XQ, WQ, x_scale, w_scale) -> List[torch.Tensor]:
    """TensorList grouped GEMM; the outputs are views into ONE flat bf16 buffer
    (fp8_rowwise_grouped_gemm.hip:528-529,553-557)."""
    _check_grouped(XQ, WQ, x_scale, w_scale)
    if len(XQ) == 0:
        return []
    return _op("f8f8bf16_rowwise_grouped", list(XQ), list(WQ), list(x_scale), list(w_scale))


def f8f8bf16_rowwise_grouped_cat(XQ, WQ, x_scale, w_scale) -> torch.Tensor:
    """Same computation, outputs concatenated along M (all groups must share N)."""
    _check_grouped(XQ, WQ, x_scale, w_scale)
    _check(len(XQ) > 0, "at least one group is required")
    return _op("f8f8bf16_rowwise_grouped_cat", list(XQ), list(WQ), list(x_scale), list(w_scale))


def f8f8bf16_rowwise_grouped_stacked(XQ, WQ, x_scale, w_scale, M_sizes) -> torch.Tensor:
    """XQ [total_M, K], WQ [G, N, K], x_scale [total_M], w_scale [G, N], M_sizes int64 [G] on the GPU
    (fp8_rowwise_grouped_gemm.hip:607-655).  M_sizes is never read on the host."""
    _check(XQ.is_cuda, "XQ/WQ must be contiguous GPU tensors")
    return _op("f8f8bf16_rowwise_grouped_stacked", XQ, WQ, x_scale, w_scale, M_sizes)


def f8f8bf16_rowwise_grouped_mm(XQ, WQ, x_scale, w_scale, offsets, output) -> torch.Tensor:
    """Grouped GEMM in the torch._grouped_mm convention (fp8_rowwise_grouped_gemm.hip:720-845): the
    ranks of XQ / WQ select which dimension varies per group, `offsets` (int32, on the GPU, never
    read on the host) holds the cumulative group ends along it, and the result is written into
    `output`, which is returned.

      XQ [total_M, K], WQ [G, N, K]   offsets over M   output [total_M, N]
      XQ [G, M, K],    WQ [total_N, K] offsets over N   output [M, total_N]
      XQ [G, M, K],    WQ [G, N, K]    no offsets       output [G, M, N]
      XQ [M, total_K], WQ [N, total_K] offsets over K   output [G, M, N]
    """
    _check(XQ.is_cuda, "XQ/WQ must be contiguous GPU tensors")
    return _op("f8f8bf16_rowwise_grouped_mm", XQ, WQ, x_scale, w_scale, offsets, output)


def f8f8bf16_rowwise_grouped_dynamic(XQ, WQ, x_scale, w_scale, zero_start_index_M, zeroing_output_tensor=True) -> torch.Tensor:
    """XQ [G, M, K], WQ [G, N, K] -> bf16 [G, M, N]; only the first zero_start_index_M[g] rows of group
    g are computed, the others are zero (or uninitialised when zeroing_output_tensor is False).
    Deprecated in the reference (fp8_rowwise_grouped_gemm.hip:656-714) but still registered."""
    _check(XQ.dim() == 3, "Input XQ must be 3D (G,M,K).")
    _check(WQ.dim() == 3, "Input WQ must be 3D (G,N,K).")
    _check(XQ.is_cuda and XQ.is_contiguous() and WQ.is_cuda and WQ.is_contiguous(), "XQ/WQ must be contiguous GPU tensors")
    _check(XQ.dtype == WQ.dtype, f"XQ and WQ dtypes must match, got {XQ.dtype} vs {WQ.dtype}")
    _check(XQ.dtype == FP8_DTYPE, f"XQ and WQ must be {FP8_DTYPE} on gfx950, got {XQ.dtype}")
    _check(x_scale.dtype == torch.float32 and w_scale.dtype == torch.float32, "Scales must be float32.")
    G, M, K = XQ.shape
    N = WQ.shape[1]
    _check(WQ.shape[0] == G and x_scale.numel() == G * M and w_scale.numel() == G * N and WQ.shape[2] == K,
           "All inputs must have the same number of groups.")
    _check(N >= 512 and K >= 512, "N and K must be at least 512 for grouped gemm. For smaller inputs, consider unrolling.")
    zs = zero_start_index_M
    _check(zs.is_cuda and zs.dtype == torch.int64 and zs.numel() == G, "zero_start_index_M must be an int64 GPU tensor with G entries")
    _check(WQ.device == XQ.device and x_scale.device == XQ.device and w_scale.device == XQ.device and zs.device == XQ.device,
           "all operands must be on the same device")
    Y = torch.empty((G, M, N), dtype=torch.bfloat16, device=XQ.device)
    if Y.numel() == 0:
        return Y
    xs, ws, zs = x_scale.contiguous(), w_scale.contiguous(), zs.contiguous()
    with _on_device(XQ.device):
        _lib.check(_lib.lib().mslk_amd_f8f8bf16_rowwise_grouped_dynamic(
            XQ.data_ptr(), WQ.data_ptr(), xs.data_ptr(), ws.data_ptr(), zs.data_ptr(), G, M, N, K, Y.data_ptr(),
            1 if zeroing_output_tensor else 0, _stream_ptr(XQ.device)))
    return Y


def f8f8bf16_rowwise_batched(XQ, WQ, x_scale, w_scale, bias=None, use_fast_accum=True, output=None) -> torch.Tensor:
    """XQ [B, M, K], WQ [B, N, K], x_scale [B, M], w_scale [B, N] -> bf16 [B, M, N]
    (fp8_rowwise_batched_gemm.hip:199-254).  `bias` [B, N] (fp32 or bf16) is added per batch as the
    reference's CUTLASS build does (f8f8bf16_rowwise_batched_common.cuh:272-275); its ROCm build
    accepts the argument and drops it."""
    _check(XQ.dim() == 3 and WQ.dim() == 3, "Inputs must have 3 dimensions, with the first being batch.")
    _check(XQ.dtype == WQ.dtype, f"XQ and WQ dtypes must match, got {XQ.dtype} vs {WQ.dtype}")
    _check(XQ.dtype == FP8_DTYPE, f"XQ and WQ must be {FP8_DTYPE} on gfx950, got {XQ.dtype}")
    _check(x_scale.dtype == torch.float32 and w_scale.dtype == torch.float32, "Scales must be float32.")
    _check(use_fast_accum, "AMD does not support disabling use_fast_accum.")
    _check(XQ.is_cuda and XQ.is_contiguous(), "XQ must be a contiguous GPU tensor")
    _check(WQ.is_cuda and WQ.is_contiguous(), "WQ must be a contiguous GPU tensor")
    B, M, K = XQ.shape
    N = WQ.shape[1]
    _check(WQ.shape[0] == B and WQ.shape[2] == K, "XQ must be (B, M, K) and WQ (B, N, K)")
    _check(x_scale.numel() == B * M and w_scale.numel() == B * N, "scale sizes must match B*M and B*N")
    _check(WQ.device == XQ.device and x_scale.device == XQ.device and w_scale.device == XQ.device,
           "all operands must be on the same device")
    if output is not None:
        Y = output
        _check(Y.dim() == 3, "Output tensor must have three dimensions.")
        _check(tuple(Y.shape) == (B, M, N), "output has the wrong shape")
        _check(Y.dtype == torch.bfloat16, "output must be bfloat16")
        _check(Y.is_cuda and Y.is_contiguous() and Y.device == XQ.device, "output must be a contiguous GPU tensor")
    else:
        Y = torch.empty((B, M, N), dtype=torch.bfloat16, device=XQ.device)
    if Y.numel() == 0:
        return Y
    xs, ws = x_scale.contiguous(), w_scale.contiguous()
    bias_ptr, bias_code, _keep = _bias_args(bias, B * N, XQ.device)
    with _on_device(XQ.device):
        _lib.check(_lib.lib().mslk_amd_f8f8bf16_rowwise_batched(
            XQ.data_ptr(), WQ.data_ptr(), xs.data_ptr(), ws.data_ptr(), bias_ptr, bias_code, B, M, N, K,
            Y.data_ptr(), _stream_ptr(XQ.device)))
    return Y


# ---------------------------------------------------------------------------------------------
# registration
# ---------------------------------------------------------------------------------------------
# GPU kernels that are Python functions; every other operator's kernel is native.
_PYTHON_IMPLS = {
    "f8f8bf16_rowwise_grouped_dynamic": f8f8bf16_rowwise_grouped_dynamic,
    "f8f8bf16_rowwise_batched": f8f8bf16_rowwise_batched,
}


def _fake_quantize_rowwise(X, WQ, w_scale, bias=None):
    return (torch.empty(tuple(X.shape[:-1]) + (WQ.shape[0],), dtype=torch.bfloat16, device=X.device),
            torch.empty(X.shape, dtype=FP8_DTYPE, device=X.device),
            torch.empty(X.shape[:-1], dtype=torch.float32, device=X.device))


def _fake_rowwise(XQ, WQ, x_scale, w_scale, bias=None, use_fast_accum=True):
    # mslk/gemm/_meta.py:26-50, generalised to any number of leading dims
    return torch.empty(tuple(XQ.shape[:-1]) + (WQ.shape[0],), dtype=torch.bfloat16, device=XQ.device)


def _fake_rowwise_f16(XQ, WQ, x_scale, w_scale, bias=None, use_fast_accum=True):
    # mslk/gemm/_meta.py:516-529, generalised to any number of leading dims
    return torch.empty(tuple(XQ.shape[:-1]) + (WQ.shape[0],), dtype=torch.float16, device=XQ.device)


def _fake_rowwise_out(XQ, WQ, x_scale, w_scale, output, bias=None, use_fast_accum=True):
    return None


def _fake_grouped(XQ, WQ, x_scale, w_scale):
    # as the kernel (and the reference): views into one flat buffer
    if len(XQ) == 0:
        return []
    sizes = [x.shape[0] * w.shape[0] for x, w in zip(XQ, WQ)]
    flat = torch.empty(sum(sizes), dtype=torch.bfloat16, device=XQ[0].device)
    return [t.view(x.shape[0], w.shape[0]) for t, x, w in zip(flat.split(sizes), XQ, WQ)]


def _fake_grouped_cat(XQ, WQ, x_scale, w_scale):
    return torch.empty((sum(x.shape[0] for x in XQ), WQ[0].shape[0]), dtype=torch.bfloat16, device=XQ[0].device)


def _fake_grouped_stacked(XQ, WQ, x_scale, w_scale, M_sizes):
    # mslk/gemm/_meta.py:114-126
    return torch.empty((XQ.shape[0], WQ.shape[1]), dtype=torch.bfloat16, device=XQ.device)


def _fake_grouped_dynamic(XQ, WQ, x_scale, w_scale, zero_start_index_M, zeroing_output_tensor=True):
    return torch.empty((XQ.shape[0], XQ.shape[1], WQ.shape[1]), dtype=torch.bfloat16, device=XQ.device)


def _fake_grouped_mm(XQ, WQ, x_scale, w_scale, offsets, output):
    return output


def _fake_batched(XQ, WQ, x_scale, w_scale, bias=None, use_fast_accum=True, output=None):
    # mslk/gemm/_meta.py:68-83
    if output is not None:
        return output
    return torch.empty((XQ.shape[0], XQ.shape[1], WQ.shape[1]), dtype=torch.bfloat16, device=XQ.device)


_FAKES = {
    "f8f8bf16_rowwise": _fake_rowwise,
    "f8f8bf16_rowwise_out": _fake_rowwise_out,
    "f8f8f16_rowwise": _fake_rowwise_f16,
    "f8f8bf16_rowwise_preshuffle": _fake_rowwise,
    "f8f8f16_rowwise_preshuffle": _fake_rowwise_f16,
    "f8f8bf16_rowwise_grouped": _fake_grouped,
    "f8f8bf16_rowwise_grouped_cat": _fake_grouped_cat,
    "f8f8bf16_rowwise_grouped_stacked": _fake_grouped_stacked,
    "f8f8bf16_rowwise_grouped_dynamic": _fake_grouped_dynamic,
    "f8f8bf16_rowwise_grouped_mm": _fake_grouped_mm,
    "f8f8bf16_rowwise_batched": _fake_batched,
    "quantize_f8f8bf16_rowwise": _fake_quantize_rowwise,
}


def _register() -> None:
    for name, schema in _SCHEMAS.items():
        if not hasattr(torch.ops.mslk, name):
            _library.define(name + schema)
            torch.library.register_fake(f"mslk::{name}", _FAKES[name], lib=_library)
    for name, impl in _PYTHON_IMPLS.items():
        # GPU kernel: on ROCm builds of PyTorch HIP tensors dispatch on the "CUDA" key.
        _library.impl(name, impl, "CUDA", allow_override=True)


_register()
