"""Tensors whose rows or chunks are more than one dimension of a launch may hold: the grid goes on along y, or every lane walks
several chunks.  Compared with the same rows in slices that need neither."""
import pytest
import torch

import mslk_amd

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
GRID_X = 1 << 21   # workgroups along x (csrc/rows.h)


def _slices(rows, step=GRID_X // 4):
    return [slice(b, min(b + step, rows)) for b in range(0, rows, step)]


@pytest.mark.parametrize("K,per_workgroup", [(2568, 1), (1032, 4)])
def test_quantizer_with_more_workgroups_than_one_line_of_the_grid(K, per_workgroup):
    rows = GRID_X * per_workgroup + 3 * per_workgroup + (1 if per_workgroup > 1 else 0)
    x = torch.randn(rows, K, device=DEV, dtype=torch.bfloat16)
    q, s = mslk_amd.quantize_fp8_row(x)
    for part in _slices(rows):
        want, want_scale = mslk_amd.quantize_fp8_row(x[part])
        assert torch.equal(q[part].view(torch.uint8), want.view(torch.uint8)) and torch.equal(s[part], want_scale)


def test_gated_product_with_more_workgroups_than_one_line_of_the_grid():
    rows, D = GRID_X + 3, 2056
    x = torch.randn(rows, 2 * D, device=DEV, dtype=torch.bfloat16)
    q, s = mslk_amd.silu_mul_quant(x[:, :D], x[:, D:])
    for part in _slices(rows):
        want, want_scale = mslk_amd.silu_mul_quant(x[part, :D], x[part, D:])
        assert torch.equal(q[part].view(torch.uint8), want.view(torch.uint8)) and torch.equal(s[part], want_scale)


def test_dequantizer_beyond_two_to_the_31_chunks():
    K = 56   # seven chunks of eight codes
    rows = ((1 << 31) + 7) // 7 + 5
    one = torch.randint(0, 0x78, (1 << 20,), device=DEV, dtype=torch.uint8)
    codes = one.repeat(rows * K // one.numel() + 1)[: rows * K].view(rows, K).view(mslk_amd.FP8_DTYPE)
    s = torch.rand(rows, device=DEV) + 0.5
    y = mslk_amd.dequantize_fp8_row(codes, s)
    for part in _slices(rows, 1 << 25):
        assert torch.equal(y[part].view(torch.int16), mslk_amd.dequantize_fp8_row(codes[part], s[part]).view(torch.int16))
    del y, codes
    torch.cuda.empty_cache()
