"""The package's own functions, as a program calls them instead of the operators: traced, beside autograd, on CPU tensors and
without a build.  CPU; tensors of a GPU are fake ones, which have shapes and no data."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

import mslk_amd

F8, BF16, DEV = torch.float8_e4m3fn, torch.bfloat16, "cuda"
ROWWISE = ["f8f8bf16_rowwise", "f8f8f16_rowwise", "f8f8bf16_rowwise_preshuffle", "f8f8f16_rowwise_preshuffle"]


def _empty(*shape, dtype=torch.float32, grad=False):
    return torch.empty(*shape, dtype=dtype, device=DEV, requires_grad=grad)


def test_results_and_written_outputs_stay_outside_of_autograd():
    """A scale that requires a gradient (the quantizer's, of an input that does) makes no graph of a product."""
    with FakeTensorMode():
        wq, ws = _empty(4, 768, 512, dtype=F8), _empty(4, 768)
        xq, xs = _empty(40, 512, dtype=F8), _empty(40, grad=True)
        out = _empty(40, 768, dtype=BF16)
        results = [
            *mslk_amd.quantize_f8f8bf16_rowwise(_empty(3, 512, dtype=BF16, grad=True), wq[0], ws[0]),
            *mslk_amd.f8f8bf16_rowwise_grouped([xq, xq], [wq[0], wq[1]], [xs, xs], [ws[0], ws[1]]),
            mslk_amd.f8f8bf16_rowwise_grouped_cat([xq, xq], [wq[0], wq[1]], [xs, xs], [ws[0], ws[1]]),
            mslk_amd.f8f8bf16_rowwise_grouped_stacked(xq, wq, xs, ws, _empty(4, dtype=torch.int64)),
            mslk_amd.f8f8bf16_rowwise_grouped_mm(xq, wq, xs, ws, _empty(4, dtype=torch.int32), out),
        ]
        assert results[-1] is out and not any(r.requires_grad for r in results)
