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


@pytest.mark.parametrize("name", ROWWISE + ["f8f8bf16_rowwise_out"])
def test_dense_functions_trace_to_their_operator(name):
    from torch.fx.experimental.proxy_tensor import make_fx
    function = getattr(mslk_amd, name)

    def call(xq, wq, xs, ws):
        if name.endswith("_out"):
            out = xq.new_empty(xq.shape[0], wq.shape[0], dtype=BF16)
            function(xq, wq, xs, ws, out)
            return out
        return function(xq, wq, xs, ws)

    with FakeTensorMode():
        args = (_empty(64, 128, dtype=F8), _empty(256, 128, dtype=F8), _empty(64, grad=True), _empty(256))
        y = call(*args)
        assert y.shape == (64, 256) and y.dtype == (torch.float16 if name.startswith("f8f8f16") else BF16)
        assert not y.requires_grad
        graph = make_fx(call)(*args).graph
    assert [n.target for n in graph.nodes if "mslk" in str(n.target)] == [getattr(torch.ops.mslk, name).default]


def test_cpu_tensors_are_refused_as_the_kernel_would():
    xq, wq, xs, ws = torch.zeros(4, 512).to(F8), torch.zeros(8, 512).to(F8), torch.ones(4), torch.ones(8)
    for name in ROWWISE:
        with pytest.raises(RuntimeError, match="XQ must be a contiguous GPU tensor"):
            getattr(mslk_amd, name)(xq, wq, xs, ws)
    for call, message in [
        (lambda: mslk_amd.f8f8bf16_rowwise_out(xq, wq, xs, ws, torch.empty(4, 8, dtype=BF16)), "XQ must be a contiguous GPU tensor"),
        (lambda: mslk_amd.quantize_f8f8bf16_rowwise(torch.zeros(4, 512, dtype=BF16), wq, ws), "WQ must be a contiguous 2-D GPU tensor"),
        (lambda: mslk_amd.f8f8bf16_rowwise_grouped([xq], [wq], [xs], [ws]), "XQ tensors must be contiguous GPU tensors"),
        (lambda: mslk_amd.f8f8bf16_rowwise_grouped([], [wq], [], []), "same number of groups"),
        (lambda: mslk_amd.f8f8bf16_rowwise_grouped_cat([], [], [], []), "at least one group"),
        (lambda: mslk_amd.f8f8bf16_rowwise_grouped_stacked(xq, wq[None], xs, ws, torch.tensor([4])), "XQ/WQ must be contiguous GPU"),
        (lambda: mslk_amd.f8f8bf16_rowwise_grouped_mm(xq, wq[None], xs, ws, None, torch.empty(4, 8)), "XQ/WQ must be contiguous GPU"),
    ]:
        with pytest.raises(RuntimeError, match=message):
            call()
    assert mslk_amd.f8f8bf16_rowwise_grouped([], [], [], []) == []


@pytest.mark.gpu
@pytest.mark.parametrize("name", ROWWISE + ["f8f8bf16_rowwise_out"])
def test_dense_functions_compile_into_one_graph(name):
    function = getattr(mslk_amd, name)
    w = torch.randn(96, 256, device="cuda:0", dtype=BF16)
    wq, ws = mslk_amd.quantize_fp8_row(w)
    if "preshuffle" in name:
        wq = mslk_amd.preshuffle_b_mfma(wq)

    def linear(x):
        xq, xs = mslk_amd.quantize_fp8_row(x)
        if name.endswith("_out"):
            y = torch.empty(x.shape[0], 96, device=x.device, dtype=BF16)
            function(xq, wq, xs, ws, y)
            return y
        return function(xq, wq, xs, ws)

    x = torch.randn(40, 256, device="cuda:0", dtype=BF16)
    assert torch.equal(torch.compile(linear, backend="aot_eager", fullgraph=True)(x), linear(x))


@pytest.mark.parametrize("name,args", [
    ("mslk::silu_mul_quant", lambda: (torch.zeros(2, 8, dtype=BF16), torch.zeros(2, 8, dtype=BF16))),
    ("mslk::gather_scale_quant_dense_tokens", lambda: (torch.zeros(2, 8, dtype=BF16), torch.zeros(2, dtype=torch.int32),
                                                       torch.zeros(2, dtype=torch.int32), torch.zeros(2, 3))),
    ("triton::quantize_fp8_row", lambda: (torch.zeros(2, 8, dtype=BF16),)),
])
def test_kernels_refuse_cpu_inputs_that_reach_them(name, args):
    """An optional operand on a GPU is enough to pick the GPU's kernel; here it is called directly."""
    namespace, operator = name.split("::")
    overload = getattr(getattr(torch.ops, namespace), operator).default
    optional = [a.default_value for a in overload._schema.arguments[len(args()):]]
    with pytest.raises(RuntimeError, match="must be (a )?GPU tensor"):
        overload.redispatch(torch._C.DispatchKeySet(torch._C.DispatchKey.CUDA), *args(), *optional)


@pytest.mark.gpu
@pytest.mark.parametrize("elsewhere", ["x_scale", "w_scale"])
def test_stacked_form_refuses_scales_in_host_memory(elsewhere):
    operands = {"XQ": torch.zeros(8, 512, device="cuda:0").to(F8), "WQ": torch.zeros(2, 512, 512, device="cuda:0").to(F8),
                "x_scale": torch.ones(8, device="cuda:0"), "w_scale": torch.ones(2, 512, device="cuda:0"),
                "M_sizes": torch.tensor([3, 5], device="cuda:0")}
    operands[elsewhere] = operands[elsewhere].cpu()
    with pytest.raises(RuntimeError, match="same device"):
        torch.ops.mslk.f8f8bf16_rowwise_grouped_stacked(**operands)
