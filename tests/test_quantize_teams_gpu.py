"""The quantizer gives a row to 8 ... 1024 lanes with one to eight vectors each: row lengths on both sides of every step of
that dispatch, row counts on both sides of the one that switches to several rows per wavefront, with special rows, strided
input, padded and jagged output.  Codes and scales are the oracle's bits in both arithmetics."""
import pytest
import torch

import mslk_amd
from oracle import fp8_rowwise_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _check(got, want, what):
    (q, s), (rq, rs) = got, want
    q, rq = q.cpu().view(torch.uint8), rq.view(torch.uint8)
    nan = (rq & 0x7F) == 0x7F          # the sign of a NaN code is not part of the contract
    assert torch.equal(q[~nan], rq[~nan]) and ((q[nan] & 0x7F) == 0x7F).all(), f"codes, {what}"
    s, bad = s.cpu(), torch.isnan(rs)
    assert torch.equal(s[~bad], rs[~bad]) and torch.isnan(s[bad]).all(), f"scales, {what}"


def _rows(rows, K, dtype, g, special):
    x = torch.randn(rows, K + 8, generator=g).to(dtype)[:, :K]    # rows 16 (fp32: 32) bytes apart from contiguous
    x[0, -1] = 300.0      # the maximum in the last vector of the row
    x[1] = 0.0
    x[1, ::2] = -0.0      # zeros keep their sign
    if special:           # (the saturating arithmetic turns NaN quotients into -448 where torch.clamp keeps them)
        x[2, K // 2] = float("inf")
        x[3, K - 3] = float("nan")
    return x


SMALL = [8, 64, 72, 128, 136, 256, 264, 512, 520, 1024, 1032, 2048]
LARGE = [2056, 4096, 4104, 8192, 8200, 16384, 16392, 32768, 32776, 65536, 65544]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,Ks", [(2051, SMALL), (2051, [2056, 2560, 2568]), (2047, SMALL[:6]), (5, SMALL + LARGE)])
def test_row_lengths_around_every_step_of_the_dispatch(rows, Ks, dtype):
    g = torch.Generator().manual_seed(rows)
    for K in Ks:
        for triton in (True, False):
            x = _rows(rows, K, dtype, g, special=not triton)
            want = O.quantize_fp8_row_triton_arithmetic(x) if triton else O.quantize_fp8_row(x)
            full = torch.zeros(rows, K + 8, dtype=dtype)
            full[:, :K] = x
            got = mslk_amd.quantize_fp8_row(full.to(DEV)[:, :K], use_triton=triton)
            _check(got, want, f"{rows} x {K} {dtype} triton={triton}")


@pytest.mark.parametrize("rows,K", [(2051, 64), (2051, 520), (2051, 1024), (2051, 2048), (300, 520), (5, 65544)])
def test_rows_in_reverse_order_through_the_c_abi(rows, K):
    """A negative row stride, from the last row on: several rows of a wavefront, a wavefront or a workgroup per row."""
    from mslk_amd import _lib
    x = torch.randn(rows, K, device=DEV).bfloat16()
    q, s = torch.empty(rows, K, dtype=torch.uint8, device=DEV), torch.empty(rows, device=DEV)
    _lib.check(_lib.lib().mslk_amd_quantize_fp8_row(x[-1].data_ptr(), 0, rows, K, -K, q.data_ptr(), K, s.data_ptr(), None,
                                                    torch.cuda.current_stream().cuda_stream))
    want, want_scale = mslk_amd.quantize_fp8_row(x.flip(0), use_triton=False)
    assert torch.equal(q, want.view(torch.uint8)) and torch.equal(s, want_scale)


@pytest.mark.parametrize("groups,per_group,K", [(500, 5, 120), (3, 7, 4104), (130, 16, 1000)])
def test_dead_rows_and_padding_columns(groups, per_group, K):
    """Several rows of a wavefront with different live counts; columns up to the next multiple of 128 are zero."""
    g = torch.Generator().manual_seed(K)
    x = torch.randn(groups, per_group, K, generator=g).bfloat16()
    live = torch.randint(0, per_group + 1, (groups,), generator=g)
    q, s = mslk_amd.quantize_fp8_row(x.to(DEV), zero_start_index_M=live.to(DEV), align_rows_to=128)
    dead = torch.arange(per_group)[None, :] >= live[:, None]
    rq, rs = O.quantize_fp8_row_triton_arithmetic(x.masked_fill(dead[..., None], 0.0))
    q = q.cpu().view(torch.uint8)
    assert torch.equal(q[..., :K], rq.view(torch.uint8)) and not q[..., K:].any()
    assert torch.equal(s.cpu(), rs)


@pytest.mark.parametrize("groups,per_group,K", [(700, 3, 64), (400, 6, 264), (300, 7, 1024), (3, 7, 4104), (3, 7, 65544), (5, 4, 100)])
@pytest.mark.parametrize("triton", [True, False])
def test_dead_rows_are_zero_codes_whatever_scale_ub_is(groups, per_group, K, triton):
    """A bound of zero or below makes the scale zero or negative: 0 / 0 and 0 times a negative factor are no zero codes."""
    g = torch.Generator().manual_seed(K)
    x = torch.randn(groups, per_group, K, generator=g).bfloat16().to(DEV)
    live = torch.randint(0, per_group + 1, (groups,), generator=g)
    live[0] = 0
    dead = torch.arange(per_group)[None, :] >= live[:, None]
    for bound in (0.0, -1.0):
        q, _ = mslk_amd.quantize_fp8_row(x, torch.tensor([bound], device=DEV), live.to(DEV), triton, None, 128)
        q = q.cpu().view(torch.uint8)
        assert not q[dead].any() and not q[..., K:].any(), (bound, K)


@pytest.mark.parametrize("rows,K", [(1, 8), (300, 8), (257, 24), (1000, 576), (3, 65544), (129, 1000), (70001, 16)])
def test_dequantized_rows_take_their_own_scale(rows, K):
    """The row of a chunk comes from a multiply and a shift: chunk counts per row of one, a power of two and neither."""
    g = torch.Generator().manual_seed(rows + K)
    q = torch.randint(0, 0x7E, (rows, K), generator=g, dtype=torch.uint8).view(torch.float8_e4m3fn)
    s = torch.rand(rows, generator=g) + 0.5
    y = mslk_amd.dequantize_fp8_row(q.to(DEV), s.to(DEV))
    assert torch.equal(y.cpu(), O.dequantize_fp8_row_bf16(q, s))
