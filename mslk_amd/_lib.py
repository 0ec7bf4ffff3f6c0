"""ctypes binding of libmslk_amd.so (the C ABI declared in include/mslk_amd.h).

There is no fallback: if the shared library has not been built, `lib()` raises.
"""
from __future__ import annotations

import ctypes
import os
from ctypes import c_char_p, c_float, c_int, c_int64, c_size_t, c_void_p, POINTER

_HERE = os.path.dirname(os.path.abspath(__file__))
# MSLK_AMD_LIBRARY overrides the location of the built library (e.g. an out-of-tree build).
LIB_PATH = os.environ.get("MSLK_AMD_LIBRARY") or os.path.join(_HERE, "libmslk_amd.so")

# The operators as native PyTorch kernels on top of it (csrc/torch_ops.cpp).
TORCH_OPS_PATH = os.path.join(_HERE, "_torch_ops.so")

_lib = None

# name -> (restype, argtypes); mirrors include/mslk_amd.h one to one
SIGNATURES = {
    "mslk_amd_version": (c_char_p, []),
    "mslk_amd_last_error": (c_char_p, []),
    "mslk_amd_quantize_fp8_row": (c_int, [c_void_p, c_int, c_int64, c_int64, c_int64, c_void_p, c_int64,
                                          c_void_p, c_void_p, c_void_p]),
    "mslk_amd_quantize_fp8_row_jagged": (c_int, [c_void_p, c_int, c_int64, c_int64, c_int64, c_void_p, c_int64,
                                                 c_void_p, c_void_p, c_void_p, c_int, c_int64, c_void_p]),
    "mslk_amd_quantize_fp8_row_triton_arithmetic": (c_int, [c_void_p, c_int, c_int64, c_int64, c_int64, c_void_p, c_int64,
                                                            c_void_p, c_void_p, c_float, c_void_p, c_int, c_int64, c_void_p]),
    "mslk_amd_silu_mul_quant": (c_int, [c_void_p, c_void_p, c_int, c_int64, c_int64, c_int64, c_int64, c_void_p, c_void_p,
                                        c_void_p, c_void_p, c_int, c_void_p]),
    "mslk_amd_gather_scale_quant_dense_tokens": (c_int, [c_void_p, c_int, c_int64, c_int64, c_void_p, c_int, c_void_p, c_int,
                                                         c_int64, c_void_p, c_int, c_int64, c_int64, c_int64, c_void_p,
                                                         c_void_p, c_void_p, c_void_p, c_int, c_void_p]),
    "mslk_amd_dequantize_fp8_row": (c_int, [c_void_p, c_void_p, c_int64, c_int64, c_void_p, c_void_p]),
    "mslk_amd_f8f8bf16_rowwise": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p,
                                          c_int64, c_int64, c_int64, c_void_p, c_size_t, c_void_p]),
    "mslk_amd_f8f8bf16_rowwise_static_scratch": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p,
                                                         c_int64, c_int64, c_int64, c_void_p]),
    "mslk_amd_static_scratch_bytes": (c_size_t, []),
    "mslk_amd_quantize_f8f8bf16_rowwise": (c_int, [c_void_p, c_int, c_int64, c_void_p, c_void_p, c_void_p, c_int, c_void_p,
                                                   c_int64, c_int64, c_int64, c_void_p, c_void_p, c_void_p]),
    "mslk_amd_quantize_f8f8bf16_rowwise_supported": (c_int, [c_int64, c_int64, c_int64]),
    "mslk_amd_f8f8f16_rowwise": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p,
                                         c_int64, c_int64, c_int64, c_void_p, c_size_t, c_void_p]),
    "mslk_amd_f8f8_rowwise_preshuffle": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_int,
                                                 c_int64, c_int64, c_int64, c_void_p]),
    "mslk_amd_f8f8_rowwise_preshuffle_workspace": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_int,
                                                           c_int64, c_int64, c_int64, c_void_p, c_size_t, c_void_p]),
    "mslk_amd_preshuffle_b": (c_int, [c_void_p, c_void_p, c_int64, c_int64, c_int64, c_void_p]),
    "mslk_amd_f8f8bf16_rowwise_workspace_bytes": (c_size_t, [c_int64, c_int64, c_int64]),
    "mslk_amd_f8f8bf16_rowwise_grouped": (c_int, [c_int, POINTER(c_void_p), POINTER(c_void_p), POINTER(c_void_p),
                                                  POINTER(c_void_p), POINTER(c_void_p), POINTER(c_int64),
                                                  POINTER(c_int64), POINTER(c_int64), c_void_p]),
    "mslk_amd_f8f8bf16_rowwise_grouped_stacked": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int,
                                                          c_int64, c_int64, c_int64, c_void_p, c_void_p]),
    "mslk_amd_f8f8bf16_rowwise_grouped_mm": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int,
                                                     c_int64, c_int64, c_int64, c_void_p, c_void_p]),
    "mslk_amd_f8f8bf16_rowwise_grouped_dynamic": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int,
                                                          c_int64, c_int64, c_int64, c_void_p, c_int, c_void_p]),
    "mslk_amd_f8f8bf16_rowwise_batched": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int64,
                                                  c_int64, c_int64, c_int64, c_void_p, c_void_p]),
    "mslk_amd_debug_cast_e4m3fn": (c_int, [c_void_p, c_int64, c_void_p, c_void_p]),
    "mslk_amd_debug_dispatch_name": (c_char_p, [c_int64, c_int64, c_int64, c_int, c_int, c_int, c_int]),
    "mslk_amd_debug_grouped_dispatch_name": (c_char_p, [c_int, c_int, c_int64, c_int64, c_int64]),
    "mslk_amd_debug_grouped_list_dispatch_name": (c_char_p, [c_int, POINTER(c_int64), POINTER(c_int64), POINTER(c_int64)]),
    "mslk_amd_debug_row_walk": (c_int, [c_int, c_int, c_int, c_int, POINTER(c_int), POINTER(c_int)]),
    "mslk_amd_debug_stream_read": (c_int, [c_void_p, c_int64, c_int, c_int, c_void_p, c_void_p]),
    "mslk_amd_debug_mfma_loop": (c_int, [c_void_p, c_int, c_int, c_int, c_void_p, c_void_p]),
    "mslk_amd_debug_tile_streams": (c_int, [c_void_p, c_int64, c_void_p, c_int64, c_int64, c_int, c_int, c_int, c_void_p]),
    "mslk_amd_debug_gemm_phases": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_int64, c_int64, c_void_p, c_void_p]),
}


def _missing(path: str) -> RuntimeError:
    return RuntimeError(f"mslk_amd: {path} is missing. Build it with `python -m mslk_amd.build` "
                        "(hipcc --offload-arch=gfx950); there is no CPU or PyTorch fallback.")


def lib() -> ctypes.CDLL:
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise _missing(LIB_PATH)
        L = ctypes.CDLL(LIB_PATH)
        for name, (res, args) in SIGNATURES.items():
            fn = getattr(L, name)
            fn.restype = res
            fn.argtypes = args
        _lib = L
    return _lib


def check(rc: int) -> None:
    """Turn a non-zero return code into the RuntimeError a TORCH_CHECK would have raised."""
    if rc != 0:
        raise RuntimeError(lib().mslk_amd_last_error().decode())


def _types(schema) -> tuple:
    """The types of a schema's arguments and results: what a kernel has to agree with (names and defaults do not matter)."""
    def text(values):
        return tuple(str(v.type).replace("SymInt", "int") for v in values)
    return text(schema.arguments), text(schema.returns)


def fits(name: str, schema: str) -> bool:
    """Whether the operator `name` ("namespace::operator"), which another library may have defined, takes a kernel of `schema`."""
    import torch
    namespace, operator = name.split("::")
    overload = getattr(getattr(getattr(torch.ops, namespace), operator), "default", None)
    return overload is not None and _types(overload._schema) == _types(torch._C.parse_schema(schema))


def _register_native(names) -> None:
    """Binds the native functions to the C ABI and makes them the GPU kernels of the operators `names`."""
    for path in (LIB_PATH, TORCH_OPS_PATH):
        if not os.path.exists(path):
            raise _missing(path)
    try:
        ops = ctypes.CDLL(TORCH_OPS_PATH)
    except OSError as e:   # built against another PyTorch
        raise RuntimeError(f"mslk_amd: cannot load {TORCH_OPS_PATH}: {e}") from e
    ops.mslk_amd_torch_bind.restype, ops.mslk_amd_torch_bind.argtypes = c_char_p, [c_char_p]
    ops.mslk_amd_torch_register.restype, ops.mslk_amd_torch_register.argtypes = c_char_p, [c_char_p, c_char_p]
    error = ops.mslk_amd_torch_bind(os.fsencode(LIB_PATH))
    if error is not None:
        raise RuntimeError(f"mslk_amd: cannot bind {LIB_PATH}: {error.decode()}")
    for name in names:
        error = ops.mslk_amd_torch_register(*(part.encode() for part in name.split("::")))
        if error is not None:
            raise RuntimeError(f"mslk_amd: cannot register the kernel of {name}: {error.decode()}")


def load_torch_ops(schemas, register_stub) -> None:
    """Makes the native functions the GPU kernels of the operators of `schemas` (name -> schema, all of them defined by now, by
    this package or by a library loaded before it).  An operator that was defined with other types keeps the kernel it has.
    Where the build is missing or incomplete (or another library named by MSLK_AMD_LIBRARY is), `register_stub(name, kernel)`
    is called for each instead: a kernel that tries again when it is used, and raises what is wrong."""
    import warnings
    names = []
    for name, schema in schemas.items():
        if fits(name, schema):
            names.append(name)
        else:
            warnings.warn(f"mslk_amd: {name} is already defined with other argument or result types than {schema}; its GPU "
                          "kernel stays as it is")
    try:
        _register_native(names)
    except RuntimeError:
        def stub(name):
            def kernel(*args, **kwargs):
                import torch
                _register_native(names)   # takes the place of the stubs
                namespace, operator = name.split("::")
                return getattr(getattr(torch.ops, namespace), operator)(*args, **kwargs)
            return kernel

        for name in names:
            register_stub(name, stub(name))
