"""Importing the package beside another library that defined some of its operators first: the GPU kernels are replaced where
the types agree, other operators keep what they have, and the import never takes the process down.  CPU, one process each."""
import os
import shutil
import subprocess
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _run(code, **env):
    return subprocess.run([sys.executable, "-c", code], cwd=ROOT, env={**os.environ, **env}, capture_output=True, text=True, timeout=300)


def test_operator_defined_first_with_another_result_type_keeps_its_kernel():
    r = _run('''
import warnings, torch
foreign = torch.library.Library("mslk", "FRAGMENT")
foreign.define("gather_scale_quant_dense_tokens(Tensor x, Tensor token_indices, Tensor expert_indices, Tensor scores, "
               "Tensor? scale_ub=None, Tensor? valid_token_count=None) -> Tensor")
foreign.impl("gather_scale_quant_dense_tokens", lambda *args: args[0], "CUDA")
foreign.define("silu_mul_quant(Tensor x0, Tensor x1, Tensor? scale_ub=None, Tensor? valid_token_count=None) -> (Tensor, Tensor)")
with warnings.catch_warnings(record=True) as caught:
    warnings.simplefilter("always")
    import mslk_amd
said = [str(w.message) for w in caught if "mslk_amd" in str(w.message)]
assert len(said) == 1 and "mslk::gather_scale_quant_dense_tokens" in said[0], said
assert "torch_ops" not in torch._C._dispatch_dump("mslk::gather_scale_quant_dense_tokens")
assert "CUDA: registered at torch_ops.cpp" in torch._C._dispatch_dump("mslk::silu_mul_quant")   # the same types: replaced
assert "CUDA: registered at torch_ops.cpp" in torch._C._dispatch_dump("mslk::f8f8bf16_rowwise")
print("imported")
''')
    assert r.returncode == 0 and "imported" in r.stdout, r.stderr[-3000:]


def test_operator_defined_first_by_compiled_code_gets_the_native_kernel(tmp_path):
    """A C++ kernel with the operator's schema and another C++ signature (Tensor by value)."""
    source, library = tmp_path / "first.cpp", tmp_path / "first.so"
    source.write_text('''
#include <ATen/core/Tensor.h>
#include <torch/library.h>
static at::Tensor product(at::Tensor XQ, at::Tensor, at::Tensor, at::Tensor, std::optional<at::Tensor>, bool) { return XQ; }
TORCH_LIBRARY_FRAGMENT(mslk, m) {
  m.def("f8f8bf16_rowwise(Tensor XQ, Tensor WQ, Tensor x_scale, Tensor w_scale, Tensor? bias=None, bool use_fast_accum=True) -> Tensor");
}
TORCH_LIBRARY_IMPL(mslk, CUDA, m) { m.impl("f8f8bf16_rowwise", product); }
''')
    home = os.path.dirname(torch.__file__)
    subprocess.run(["g++", "-O0", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", f"-I{home}/include",
                    f"-I{home}/include/torch/csrc/api/include", str(source), "-o", str(library), f"-L{home}/lib", "-ltorch",
                    "-ltorch_cpu", "-lc10"], check=True, timeout=300)
    r = _run(f'''
import torch
torch.ops.load_library({str(library)!r})
import mslk_amd
assert "CUDA: registered at torch_ops.cpp" in torch._C._dispatch_dump("mslk::f8f8bf16_rowwise")
print("imported")
''')
    assert r.returncode == 0 and "imported" in r.stdout, r.stderr[-3000:]


CALL = """
cuda = torch._C.DispatchKeySet(torch._C.DispatchKey.CUDA)   # the GPU's kernel, on CPU tensors
def call():
    try:
        torch.ops.mslk.f8f8bf16_rowwise.default.redispatch(cuda, *[torch.zeros(1, 16)] * 4, None, True)
    except RuntimeError as e:
        return str(e)
"""


def test_a_process_that_imported_before_the_build_finds_it_later(tmp_path):
    package = shutil.copytree(os.path.join(ROOT, "mslk_amd"), tmp_path / "mslk_amd", ignore=shutil.ignore_patterns("*.so", "csrc"))
    r = _run(f'''
import shutil, sys, torch
sys.path.insert(0, {str(tmp_path)!r})
import mslk_amd
assert mslk_amd.__file__.startswith({str(tmp_path)!r})
{CALL}
assert "libmslk_amd.so is missing" in call(), call()
shutil.copy({os.path.join(ROOT, "mslk_amd", "libmslk_amd.so")!r}, {str(package)!r})
assert "_torch_ops.so is missing" in call(), call()
shutil.copy({os.path.join(ROOT, "mslk_amd", "_torch_ops.so")!r}, {str(package)!r})
call()   # replaces the kernels and calls the operator again, which has none for the CPU
assert "must be torch.float8_e4m3fn" in call(), call()      # the native checks
print("imported")
''')
    assert r.returncode == 0 and "imported" in r.stdout, r.stderr[-3000:]


def test_a_library_without_an_entry_point_leaves_no_kernel_over_null_pointers(tmp_path):
    source, library = tmp_path / "older.c", tmp_path / "libolder.so"
    source.write_text('const char* mslk_amd_last_error(void) { return ""; }')
    subprocess.run(["gcc", "-shared", "-fPIC", str(source), "-o", str(library)], check=True)
    r = _run(f'''
import torch, mslk_amd
{CALL}
assert "cannot bind" in call() and "does not export" in call(), call()
print("imported")
''', MSLK_AMD_LIBRARY=str(library))
    assert r.returncode == 0 and "imported" in r.stdout, r.stderr[-3000:]


def test_the_c_library_alone_is_built_without_pytorch():
    make = ["make", "-n", "-B", "-C", os.path.join(ROOT, "mslk_amd", "csrc"), "PYTHON=/nonexistent"]
    r = subprocess.run(make, capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "libmslk_amd.so" in r.stdout and "torch" not in r.stdout, r.stdout[-500:] + r.stderr
