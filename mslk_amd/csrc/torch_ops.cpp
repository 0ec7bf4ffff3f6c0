// The operators of the path as native PyTorch kernels: argument checks, output and workspace allocation, and one call of
// the C ABI.  Host code only; schemas, shape functions and the operators off the hot path are in mslk_amd/*.py.
//
// Why native: at decode sizes a call is bound by the host.  The same layer in Python took 18 us per fused decode call and
// 23 us for a quantizer call and a GEMM call, whose kernels take 13.7 and 18 us (M = 1 and 16, N = K = 8192), and 50 us
// for sixteen groups passed as lists of tensors.
//
// Validation and error messages follow the reference's ROCm host wrappers
// (csrc/gemm/ck/fp8_rowwise/fp8fp8bf16_rowwise_gemm.hip:499-550,
//  csrc/gemm/ck/fp8_rowwise_grouped/fp8_rowwise_grouped_gemm.hip:481-559,607-655), except that `bias` is implemented.
#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/zeros.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/library.h>

#include <cstring>
#include <optional>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/mslk_amd.h"

namespace {

using at::Tensor;
using at::TensorList;
using OptTensor = std::optional<Tensor>;

constexpr auto kF8 = at::kFloat8_e4m3fn;

// ---------------------------------------------------------------------------------------------------------------------
// The C ABI, bound to the library that mslk_amd/_lib.py names
// ---------------------------------------------------------------------------------------------------------------------
#define MSLK_AMD_ENTRY_POINTS(X)                                                                                       \
  X(mslk_amd_last_error)                                                                                               \
  X(mslk_amd_quantize_fp8_row)                                                                                         \
  X(mslk_amd_quantize_fp8_row_jagged)                                                                                  \
  X(mslk_amd_quantize_fp8_row_triton_arithmetic)                                                                       \
  X(mslk_amd_dequantize_fp8_row)                                                                                       \
  X(mslk_amd_silu_mul_quant)                                                                                           \
  X(mslk_amd_gather_scale_quant_dense_tokens)                                                                          \
  X(mslk_amd_f8f8bf16_rowwise)                                                                                         \
  X(mslk_amd_f8f8f16_rowwise)                                                                                          \
  X(mslk_amd_f8f8_rowwise_preshuffle_workspace)                                                                        \
  X(mslk_amd_f8f8bf16_rowwise_workspace_bytes)                                                                         \
  X(mslk_amd_quantize_f8f8bf16_rowwise)                                                                                \
  X(mslk_amd_quantize_f8f8bf16_rowwise_supported)                                                                      \
  X(mslk_amd_f8f8bf16_rowwise_grouped)                                                                                 \
  X(mslk_amd_f8f8bf16_rowwise_grouped_stacked)                                                                         \
  X(mslk_amd_f8f8bf16_rowwise_grouped_mm)

struct Api {
#define X(name) decltype(&::name) name = nullptr;
  MSLK_AMD_ENTRY_POINTS(X)
#undef X
} api;   // written once, by mslk_amd_torch_bind() while the package is imported

void check_rc(int rc) {
  if (rc != 0) TORCH_CHECK(false, api.mslk_amd_last_error());
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Tensor empty_on(at::IntArrayRef sizes, at::ScalarType dtype, const Tensor& like) {
  return Tensor(at::detail::empty_cuda(sizes, dtype, like.device(), std::nullopt));
}

// A contiguous tensor with the elements of `t` (itself when it is one).
c10::MaybeOwned<Tensor> contiguous(const Tensor& t) { return t.expect_contiguous(); }

int64_t rows_of(const Tensor& t) {   // product of all dimensions but the last
  int64_t m = 1;
  for (int64_t d = 0; d + 1 < t.dim(); ++d) m *= t.size(d);
  return m;
}

at::DimVector leading(const Tensor& t, std::optional<int64_t> last = std::nullopt) {
  at::DimVector s(t.sizes().begin(), t.sizes().end() - 1);
  if (last) s.push_back(*last);
  return s;
}

bool aligned16(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0; }

struct Bias {
  c10::MaybeOwned<Tensor> keep;
  const void* ptr = nullptr;
  int code = MSLK_AMD_BIAS_NONE;
};
Bias bias_of(const OptTensor& bias, int64_t N, const Tensor& like) {
  Bias b;
  if (!bias.has_value() || !bias->defined()) return b;
  TORCH_CHECK(bias->device() == like.device(), "bias must be on the same device as XQ");
  TORCH_CHECK(bias->scalar_type() == at::kFloat || bias->scalar_type() == at::kBFloat16, "Bias type must be bfloat16 or float32 if provided.");
  TORCH_CHECK(bias->numel() == N, "bias must have N=", N, " elements, got ", bias->numel());
  b.keep = contiguous(*bias);
  b.ptr = b.keep->const_data_ptr();
  b.code = bias->scalar_type() == at::kFloat ? MSLK_AMD_BIAS_F32 : MSLK_AMD_BIAS_BF16;
  return b;
}

// ---------------------------------------------------------------------------------------------------------------------
// quantizer
// ---------------------------------------------------------------------------------------------------------------------
int float_code(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16: return MSLK_AMD_DTYPE_BF16;
    case at::kHalf: return MSLK_AMD_DTYPE_F16;
    case at::kFloat: return MSLK_AMD_DTYPE_F32;
    default: return -1;
  }
}

Tensor first_scalar(const Tensor& t) { return t.to(at::kFloat).reshape(-1).slice(0, 0, 1).contiguous(); }

// One quantizer launch.  No `triton_eps`: the arithmetic of the reference's torch branch; otherwise that of its Triton kernel
// with that lower bound of the row maximum.
std::tuple<Tensor, Tensor> quantize_launch(const Tensor& a, const OptTensor& scale_ub, const OptTensor& zero_start_index_M,
                                           std::optional<int64_t> align_rows_to, std::optional<double> triton_eps) {
  const int code = float_code(a.scalar_type());
  TORCH_CHECK(code >= 0, "quantize_fp8_row: unsupported input dtype ", a.scalar_type(), " (bf16, fp16, fp32 are supported)");
  TORCH_CHECK(a.dim() >= 1, "quantize_fp8_row: input must have at least one dimension");
  // (an optional operand on a GPU is enough to get here)
  TORCH_CHECK(a.is_cuda(), "quantize_fp8_row: input must be a GPU tensor");
  // same restriction as the reference's GPU path (fp8_quantize.py:235)
  TORCH_CHECK(a.dim() <= 4, "Only up to 4 dimension input tensor is supported if use_triton is True");
  const int64_t K = a.size(-1), rows = rows_of(a);
  TORCH_CHECK(K != 0, "quantize_fp8_row: cannot take the row maximum of an empty last dimension");
  // The kernel takes one row stride; anything else (transposed views, broadcast dims) is packed first.
  const bool strided_rows = a.dim() == 2 && a.stride(-1) == 1;
  const auto a2 = strided_rows ? c10::MaybeOwned<Tensor>::borrowed(a) : contiguous(a);
  const int64_t row_stride = strided_rows ? a.stride(0) : K;
  int64_t K_out = K;
  if (align_rows_to) {
    TORCH_CHECK(*align_rows_to != 0, "quantize_fp8_row: align_rows_to must not be zero");
    K_out = (K + *align_rows_to - 1) / *align_rows_to * *align_rows_to;
  }
  Tensor xq = empty_on(leading(a, K_out), kF8, a);
  Tensor scale = empty_on(leading(a), at::kFloat, a);
  Tensor ub;
  if (scale_ub.has_value() && scale_ub->defined()) {
    TORCH_CHECK(scale_ub->device() == a.device(), "'scale_ub' must be on the same device as 'a'");   // fp8_quantize.py:229-230
    ub = first_scalar(*scale_ub);
  }
  const float* ub_ptr = ub.defined() ? ub.const_data_ptr<float>() : nullptr;
  Tensor zs;
  int64_t rows_per_group = 1;
  int zs_code = MSLK_AMD_INDEX_I64;
  if (zero_start_index_M.has_value() && zero_start_index_M->defined()) {
    // One entry per [N, K] matrix of the input viewed as [B, M, N, K] (fp8_quantize.py:236-243).
    rows_per_group = a.dim() >= 2 ? a.size(-2) : 1;
    const Tensor& z = *zero_start_index_M;
    TORCH_CHECK(z.device() == a.device(), "'zero_start_index_M' must be on the same device as 'a'");
    TORCH_CHECK(z.scalar_type() == at::kLong || z.scalar_type() == at::kInt, "zero_start_index_M must be int64 or int32, got ", z.scalar_type());
    TORCH_CHECK(rows_per_group != 0 && z.numel() * rows_per_group == rows, "zero_start_index_M must have one entry per group of ",
                rows_per_group, " rows (", rows / std::max<int64_t>(rows_per_group, 1), " entries), got ", z.numel());
    zs = z.contiguous();
    zs_code = zs.scalar_type() == at::kLong ? MSLK_AMD_INDEX_I64 : MSLK_AMD_INDEX_I32;
  }
  if (rows == 0) return {xq, scale};
  const void* zs_ptr = zs.defined() ? zs.const_data_ptr() : nullptr;
  const c10::DeviceGuard guard(a.device());
  void* stream = stream_of(a);
  float* sc = scale.mutable_data_ptr<float>();
  const void* x = a2->const_data_ptr();
  void* out = xq.mutable_data_ptr();
  if (triton_eps)
    check_rc(api.mslk_amd_quantize_fp8_row_triton_arithmetic(x, code, rows, K, row_stride, out, K_out, sc, ub_ptr, (float)*triton_eps,
                                                             zs_ptr, zs_code, rows_per_group, stream));
  else if (zs_ptr)
    check_rc(api.mslk_amd_quantize_fp8_row_jagged(x, code, rows, K, row_stride, out, K_out, sc, ub_ptr, zs_ptr, zs_code, rows_per_group, stream));
  else
    check_rc(api.mslk_amd_quantize_fp8_row(x, code, rows, K, row_stride, out, K_out, sc, ub_ptr, stream));
  return {xq, scale};
}

// triton::quantize_fp8_row (fp8_quantize.py:319-378).  `use_triton` picks the arithmetic, as in the reference; its torch branch
// ignores `zero_start_index_M` and `align_rows_to`, here both arithmetics honour them.
std::tuple<Tensor, Tensor> quantize_fp8_row(const Tensor& a, const OptTensor& scale_ub, const OptTensor& zero_start_index_M,
                                            bool use_triton, std::optional<c10::Device> output_device,
                                            std::optional<int64_t> align_rows_to, std::optional<double> eps_opt) {
  // without eps_opt: get_fp8_constants()'s eps (mslk/utils/triton/fp8_utils.py:23-40)
  auto [q, s] = quantize_launch(a, scale_ub, zero_start_index_M, align_rows_to,
                                use_triton ? std::optional<double>(eps_opt.value_or(1e-12)) : std::nullopt);
  if (output_device && *output_device != a.device()) return {q.to(*output_device), s.to(*output_device)};
  return {q, s};
}

// mslk::quantize_fp8_per_row: always the bits of the reference's torch emulation (fp8_quantize.py:356-378).
std::tuple<Tensor, Tensor> quantize_fp8_per_row(const Tensor& input, const OptTensor& bs, const OptTensor& scale_ub,
                                                std::optional<at::ScalarType> output_dtype, bool stochastic_rounding) {
  TORCH_CHECK_NOT_IMPLEMENTED(!bs.has_value(), "quantize_fp8_per_row: `bs` is not supported");
  TORCH_CHECK_NOT_IMPLEMENTED(!stochastic_rounding, "quantize_fp8_per_row: stochastic rounding is not supported");
  TORCH_CHECK(!output_dtype || *output_dtype == kF8, "quantize_fp8_per_row: only torch.float8_e4m3fn output is supported on gfx950");
  return quantize_launch(input, scale_ub, std::nullopt, std::nullopt, std::nullopt);
}

Tensor dequantize_fp8_row(const Tensor& xq, const Tensor& x_scale) {
  TORCH_CHECK(xq.is_contiguous() && x_scale.is_contiguous(), "Input tensors must be contiguous");
  TORCH_CHECK(xq.scalar_type() == kF8, "dequantize_fp8_row: xq must be torch.float8_e4m3fn, got ", xq.scalar_type());
  TORCH_CHECK(x_scale.scalar_type() == at::kFloat && x_scale.device() == xq.device(),
              "dequantize_fp8_row: x_scale must be a float32 tensor on the device of xq");
  TORCH_CHECK(xq.dim() >= 1, "dequantize_fp8_row: xq must have at least one dimension");
  const int64_t K = xq.size(-1), rows = K ? xq.numel() / K : 0;
  TORCH_CHECK(K == 0 || x_scale.numel() == rows, "dequantize_fp8_row: x_scale must have one entry per row (", rows, "), got ", x_scale.numel());
  Tensor out = empty_on(xq.sizes(), at::kBFloat16, xq);
  if (rows > 0) {
    const c10::DeviceGuard guard(xq.device());
    check_rc(api.mslk_amd_dequantize_fp8_row(xq.const_data_ptr(), x_scale.const_data_ptr<float>(), rows, K, out.mutable_data_ptr(), stream_of(xq)));
  }
  return out;
}

// ---------------------------------------------------------------------------------------------------------------------
// fused producers
// ---------------------------------------------------------------------------------------------------------------------
int index_code(const Tensor& t) { return t.scalar_type() == at::kLong ? MSLK_AMD_INDEX_I64 : MSLK_AMD_INDEX_I32; }
bool is_index(const Tensor& t) { return t.scalar_type() == at::kLong || t.scalar_type() == at::kInt; }

struct Scalars {   // the optional device scalars of the producers
  Tensor ub;
  const float* ub_ptr = nullptr;
  const void* count_ptr = nullptr;
  int count_code = MSLK_AMD_INDEX_I64;
};
Scalars scalars_of(const OptTensor& scale_ub, const OptTensor& valid_token_count, const Tensor& like) {
  Scalars s;
  if (scale_ub.has_value() && scale_ub->defined()) {
    s.ub = first_scalar(scale_ub->to(like.device()));
    s.ub_ptr = s.ub.const_data_ptr<float>();
  }
  if (valid_token_count.has_value() && valid_token_count->defined()) {
    TORCH_CHECK(valid_token_count->device() == like.device(), "valid_token_count must be on the device of the inputs");
    TORCH_CHECK(is_index(*valid_token_count), "valid_token_count must be int32 or int64");
    TORCH_CHECK(valid_token_count->numel() >= 1, "valid_token_count must hold one element");
    s.count_ptr = valid_token_count->const_data_ptr();
    s.count_code = index_code(*valid_token_count);
  }
  return s;
}

std::tuple<Tensor, Tensor> silu_mul_quant(const Tensor& x0, const Tensor& x1, const OptTensor& scale_ub, const OptTensor& valid_token_count) {
  TORCH_CHECK(x0.dim() == 2 && x0.stride(1) == 1, "x0 must be 2-D with unit column stride");
  TORCH_CHECK(x1.dim() == 2 && x1.stride(1) == 1, "x1 must be 2-D with unit column stride");
  TORCH_CHECK(x0.sizes() == x1.sizes(), "x0 and x1 must have the same shape");
  TORCH_CHECK(x0.scalar_type() == x1.scalar_type(), "x0 and x1 must have the same dtype");
  const int code = float_code(x0.scalar_type());
  TORCH_CHECK(code == MSLK_AMD_DTYPE_BF16 || code == MSLK_AMD_DTYPE_F16, "silu_mul_quant: inputs must be bfloat16 or float16, got ", x0.scalar_type());
  TORCH_CHECK(x1.device() == x0.device(), "x0 and x1 must be on the same device");
  TORCH_CHECK(x0.is_cuda(), "silu_mul_quant: inputs must be GPU tensors");
  const int64_t T = x0.size(0), D = x0.size(1);
  Tensor out = empty_on({T, D}, kF8, x0), out_scale = empty_on({T}, at::kFloat, x0);
  if (T == 0 || D == 0) return {out, out_scale};
  const Scalars s = scalars_of(scale_ub, valid_token_count, x0);
  const c10::DeviceGuard guard(x0.device());
  check_rc(api.mslk_amd_silu_mul_quant(x0.const_data_ptr(), x1.const_data_ptr(), code, T, D, x0.stride(0), x1.stride(0), out.mutable_data_ptr(),
                                       out_scale.mutable_data_ptr<float>(), s.ub_ptr, s.count_ptr, s.count_code, stream_of(x0)));
  return {out, out_scale};
}

std::tuple<Tensor, Tensor> gather_scale_quant_dense_tokens(const Tensor& x, const Tensor& token_indices, const Tensor& expert_indices,
                                                           const Tensor& scores, const OptTensor& scale_ub, const OptTensor& valid_token_count) {
  TORCH_CHECK(x.dim() == 2 && x.is_contiguous(), "x must be a contiguous 2-D tensor");
  TORCH_CHECK(token_indices.is_contiguous() && expert_indices.is_contiguous(), "index tensors must be contiguous");
  TORCH_CHECK(token_indices.dim() == 1 && expert_indices.dim() == 1 && expert_indices.size(0) == token_indices.size(0), "index tensors must have shape (a,)");
  const int64_t T = x.size(0), D = x.size(1), a = token_indices.size(0);
  TORCH_CHECK(scores.dim() == 2 && scores.size(0) == T, "scores must have shape (T, E)");
  const int code = float_code(x.scalar_type()), score_code = float_code(scores.scalar_type());
  TORCH_CHECK(code == MSLK_AMD_DTYPE_BF16 || code == MSLK_AMD_DTYPE_F16, "gather_scale_quant_dense_tokens: x must be bfloat16 or float16, got ", x.scalar_type());
  TORCH_CHECK(score_code >= 0, "scores must be bfloat16, float16 or float32, got ", scores.scalar_type());
  TORCH_CHECK(is_index(token_indices) && is_index(expert_indices), "indices must be int32 or int64");
  TORCH_CHECK(token_indices.device() == x.device() && expert_indices.device() == x.device() && scores.device() == x.device(),
              "all operands must be on the same device");
  TORCH_CHECK(x.is_cuda(), "gather_scale_quant_dense_tokens: inputs must be GPU tensors");
  Tensor out = empty_on({a, D}, kF8, x), out_scale = empty_on({a}, at::kFloat, x);
  if (a == 0 || D == 0) return {out, out_scale};
  const Scalars s = scalars_of(scale_ub, valid_token_count, x);
  const c10::DeviceGuard guard(x.device());
  check_rc(api.mslk_amd_gather_scale_quant_dense_tokens(
      x.const_data_ptr(), code, T, D, token_indices.const_data_ptr(), index_code(token_indices), expert_indices.const_data_ptr(),
      index_code(expert_indices), a, scores.const_data_ptr(), score_code, scores.size(1), scores.stride(0), scores.stride(1),
      out.mutable_data_ptr(), out_scale.mutable_data_ptr<float>(), s.ub_ptr, s.count_ptr, s.count_code, stream_of(x)));
  return {out, out_scale};
}

// ---------------------------------------------------------------------------------------------------------------------
// dense GEMM
// ---------------------------------------------------------------------------------------------------------------------
Tensor rowwise(const Tensor& XQ, const Tensor& WQ, const Tensor& x_scale, const Tensor& w_scale, const OptTensor& bias, bool use_fast_accum,
               const OptTensor& output, bool out_f16, bool preshuffled) {
  TORCH_CHECK(XQ.scalar_type() == WQ.scalar_type(), "XQ and WQ dtypes must match, got ", XQ.scalar_type(), " vs ", WQ.scalar_type());
  TORCH_CHECK(XQ.scalar_type() == kF8, "XQ and WQ must be torch.float8_e4m3fn on gfx950, got ", XQ.scalar_type());
  TORCH_CHECK(x_scale.scalar_type() == at::kFloat && w_scale.scalar_type() == at::kFloat, "Scales must be float32.");
  TORCH_CHECK(use_fast_accum, "AMD does not support disabling use_fast_accum.");
  TORCH_CHECK(XQ.is_cuda() && XQ.is_contiguous(), "XQ must be a contiguous GPU tensor");
  TORCH_CHECK(WQ.is_cuda() && WQ.is_contiguous(), "WQ must be a contiguous GPU tensor");
  TORCH_CHECK(XQ.dim() >= 1 && WQ.dim() == 2, "XQ must be at least 1-D and WQ 2-D");
  const int64_t N = WQ.size(0), K = WQ.size(1), M = rows_of(XQ);
  TORCH_CHECK(XQ.size(-1) == K, "XQ and WQ must share K, got ", XQ.size(-1), " vs ", K);
  TORCH_CHECK(x_scale.numel() == M, "x_scale must have M=", M, " elements, got ", x_scale.numel());
  TORCH_CHECK(w_scale.numel() == N, "w_scale must have N=", N, " elements, got ", w_scale.numel());
  TORCH_CHECK(x_scale.device() == XQ.device() && w_scale.device() == XQ.device() && WQ.device() == XQ.device(), "all operands must be on the same device");
  const auto out_dtype = out_f16 ? at::kHalf : at::kBFloat16;
  const bool given = output.has_value() && output->defined();
  if (M == 0 || N == 0 || K == 0)   // empty problem: zeros of the output shape (fp8fp8bf16_rowwise_gemm.hip:531-534)
    return given ? *output : at::zeros(leading(XQ, N), XQ.options().dtype(out_dtype));
  Tensor Y;
  if (given) {
    Y = *output;
    TORCH_CHECK(Y.dim() >= 1 && rows_of(Y) == M && Y.size(-1) == N, "output has the wrong shape");
    TORCH_CHECK(Y.scalar_type() == out_dtype, "output must be ", out_dtype);
    TORCH_CHECK(Y.is_cuda() && Y.is_contiguous() && Y.device() == XQ.device(), "output must be a contiguous GPU tensor");
  } else {
    Y = empty_on(leading(XQ, N), out_dtype, XQ);
  }
  const auto xs = contiguous(x_scale), ws = contiguous(w_scale);
  const Bias b = bias_of(bias, N, XQ);
  TORCH_CHECK(!preshuffled || (N % 16 == 0 && K % 64 == 0), "pre-shuffled weights need N % 16 == 0 and K % 64 == 0, got N=", N, " K=", K);
  const c10::DeviceGuard guard(XQ.device());
  // Rows the 16-byte loads cannot fetch: room for copies with K rounded up, on which the library runs the MFMA kernels.
  // Otherwise what the library asks for: few output tiles and a long K are split along K when there is room for the fp32
  // sums of the slices.  A block of the caching allocator, so the call stays capturable.
  const size_t bytes = !preshuffled && (K % 16 != 0 || !aligned16(XQ) || !aligned16(WQ)) ? (size_t)((M + N) * ((K + 15) / 16 * 16))
                                                                                         : api.mslk_amd_f8f8bf16_rowwise_workspace_bytes(M, N, K);
  Tensor workspace;
  if (bytes) workspace = empty_on({(int64_t)bytes}, at::kByte, XQ);
  void* wsp = bytes ? workspace.mutable_data_ptr() : nullptr;
  const float *xsp = xs->const_data_ptr<float>(), *wsc = ws->const_data_ptr<float>();
  void* stream = stream_of(XQ);
  if (preshuffled) {
    check_rc(api.mslk_amd_f8f8_rowwise_preshuffle_workspace(XQ.const_data_ptr(), WQ.const_data_ptr(), xsp, wsc, b.ptr, b.code, Y.mutable_data_ptr(),
                                                            out_f16 ? MSLK_AMD_DTYPE_F16 : MSLK_AMD_DTYPE_BF16, M, N, K, wsp, bytes, stream));
  } else {
    const auto fn = out_f16 ? api.mslk_amd_f8f8f16_rowwise : api.mslk_amd_f8f8bf16_rowwise;
    check_rc(fn(XQ.const_data_ptr(), WQ.const_data_ptr(), xsp, wsc, b.ptr, b.code, Y.mutable_data_ptr(), M, N, K, wsp, bytes, stream));
  }
  return Y;
}

template <bool F16, bool PRESHUFFLED>
Tensor rowwise_op(const Tensor& XQ, const Tensor& WQ, const Tensor& x_scale, const Tensor& w_scale, const OptTensor& bias, bool use_fast_accum) {
  return rowwise(XQ, WQ, x_scale, w_scale, bias, use_fast_accum, std::nullopt, F16, PRESHUFFLED);
}

void rowwise_out_op(const Tensor& XQ, const Tensor& WQ, const Tensor& x_scale, const Tensor& w_scale, Tensor output, const OptTensor& bias,
                    bool use_fast_accum) {
  rowwise(XQ, WQ, x_scale, w_scale, bias, use_fast_accum, output, false, false);
}

// bf16 activations in, bf16 out: the torch-branch quantizer followed by the GEMM, one launch where the library supports it
// (bits of the two launches); see mslk_amd/gemm.py.
std::tuple<Tensor, Tensor, Tensor> quantize_rowwise(const Tensor& X, const Tensor& WQ, const Tensor& w_scale, const OptTensor& bias) {
  TORCH_CHECK(WQ.scalar_type() == kF8, "WQ must be torch.float8_e4m3fn on gfx950, got ", WQ.scalar_type());
  TORCH_CHECK(w_scale.scalar_type() == at::kFloat, "Scales must be float32.");
  TORCH_CHECK(X.is_cuda() && WQ.is_cuda() && WQ.is_contiguous() && WQ.dim() == 2, "WQ must be a contiguous 2-D GPU tensor");
  TORCH_CHECK(X.dim() >= 1 && X.size(-1) == WQ.size(1), "X and WQ must share K, got ", X.dim() ? X.size(-1) : 0, " vs ", WQ.size(1));
  const int64_t N = WQ.size(0), K = WQ.size(1), M = rows_of(X);
  TORCH_CHECK(w_scale.numel() == N, "w_scale must have N=", N, " elements, got ", w_scale.numel());
  TORCH_CHECK(w_scale.device() == X.device() && WQ.device() == X.device(), "all operands must be on the same device");
  if (X.scalar_type() == at::kBFloat16 && M > 0 && api.mslk_amd_quantize_f8f8bf16_rowwise_supported(M, N, K) && aligned16(WQ)) {
    const Tensor x2 = X.dim() == 2 ? X : X.reshape({M, K});
    if (x2.stride(1) == 1 && x2.stride(0) % 8 == 0 && aligned16(x2)) {
      const auto ws = contiguous(w_scale);
      const Bias b = bias_of(bias, N, X);
      Tensor Y = empty_on(leading(X, N), at::kBFloat16, X), XQ = empty_on(X.sizes(), kF8, X), x_scale = empty_on(leading(X), at::kFloat, X);
      const c10::DeviceGuard guard(X.device());
      check_rc(api.mslk_amd_quantize_f8f8bf16_rowwise(x2.const_data_ptr(), MSLK_AMD_DTYPE_BF16, x2.stride(0), WQ.const_data_ptr(),
                                                      ws->const_data_ptr<float>(), b.ptr, b.code, Y.mutable_data_ptr(), M, N, K,
                                                      XQ.mutable_data_ptr(), x_scale.mutable_data_ptr<float>(), stream_of(X)));
      return {Y, XQ, x_scale};
    }
  }
  auto [XQ, x_scale] = quantize_launch(X, std::nullopt, std::nullopt, std::nullopt, std::nullopt);
  Tensor Y = rowwise(XQ, WQ, x_scale, w_scale, bias, true, std::nullopt, false, false);
  return {Y, XQ, x_scale};
}

// ---------------------------------------------------------------------------------------------------------------------
// grouped GEMM
// ---------------------------------------------------------------------------------------------------------------------
void check_grouped(TensorList XQ, TensorList WQ, TensorList x_scale, TensorList w_scale) {
  const size_t G = XQ.size();
  TORCH_CHECK(G == WQ.size() && G == x_scale.size() && G == w_scale.size(), "All inputs must have the same number of groups.");
  if (G == 0) return;
  const auto dev = XQ[0].device();
  TORCH_CHECK(XQ[0].scalar_type() == kF8, "XQ and WQ must be torch.float8_e4m3fn on gfx950, got ", XQ[0].scalar_type());
  for (size_t g = 0; g < G; ++g) {
    const Tensor &x = XQ[g], &w = WQ[g], &xs = x_scale[g], &ws = w_scale[g];
    TORCH_CHECK(x.is_cuda() && x.is_contiguous(), "XQ tensors must be contiguous GPU tensors");
    TORCH_CHECK(w.is_cuda() && w.is_contiguous(), "WQ tensors must be contiguous GPU tensors");
    TORCH_CHECK(x.dim() == 2 && w.dim() == 2, "Inputs must be 2D.");
    TORCH_CHECK(w.scalar_type() == kF8 && x.scalar_type() == kF8, "XQ and WQ dtypes must match, got torch.float8_e4m3fn vs ",
                w.scalar_type() != kF8 ? w.scalar_type() : x.scalar_type());
    TORCH_CHECK(w.size(0) >= 512 && w.size(1) >= 512, "N and K must be at least 512 for grouped gemm. For smaller inputs, consider unrolling.");
    TORCH_CHECK(xs.scalar_type() == at::kFloat && ws.scalar_type() == at::kFloat, "Scales must be float32.");
    TORCH_CHECK(x.size(1) == w.size(1), "XQ and WQ of a group must share K");
    TORCH_CHECK(xs.numel() == x.size(0) && ws.numel() == w.size(0), "scale sizes must match M and N of their group");
    TORCH_CHECK(x.device() == dev && w.device() == dev && xs.device() == dev && ws.device() == dev, "all operands must be on the same device");
  }
}

// The groups' products, one after the other in `flat`.
void launch_grouped(TensorList XQ, TensorList WQ, TensorList x_scale, TensorList w_scale, const Tensor& flat) {
  const size_t G = XQ.size();
  std::vector<c10::MaybeOwned<Tensor>> keep;
  keep.reserve(2 * G);
  std::vector<const void*> xq(G), wq(G);
  std::vector<const float*> xs(G), ws(G);
  std::vector<void*> y(G);
  std::vector<int64_t> M(G), N(G), K(G);
  char* out = static_cast<char*>(flat.mutable_data_ptr());
  for (size_t g = 0; g < G; ++g) {
    xq[g] = XQ[g].const_data_ptr();
    wq[g] = WQ[g].const_data_ptr();
    keep.push_back(contiguous(x_scale[g]));
    xs[g] = keep.back()->const_data_ptr<float>();
    keep.push_back(contiguous(w_scale[g]));
    ws[g] = keep.back()->const_data_ptr<float>();
    M[g] = XQ[g].size(0);
    N[g] = WQ[g].size(0);
    K[g] = WQ[g].size(1);
    y[g] = out;
    out += M[g] * N[g] * 2;
  }
  const c10::DeviceGuard guard(XQ[0].device());
  check_rc(api.mslk_amd_f8f8bf16_rowwise_grouped((int)G, xq.data(), wq.data(), xs.data(), ws.data(), y.data(), M.data(), N.data(), K.data(), stream_of(XQ[0])));
}

// The outputs are views into one flat bf16 buffer (fp8_rowwise_grouped_gemm.hip:528-529,553-557).
std::vector<Tensor> grouped_op(TensorList XQ, TensorList WQ, TensorList x_scale, TensorList w_scale) {
  check_grouped(XQ, WQ, x_scale, w_scale);
  std::vector<Tensor> outs;
  const size_t G = XQ.size();
  if (G == 0) return outs;
  int64_t total = 0;
  for (size_t g = 0; g < G; ++g) total += XQ[g].size(0) * WQ[g].size(0);
  const Tensor flat = empty_on({total}, at::kBFloat16, XQ[0]);
  launch_grouped(XQ, WQ, x_scale, w_scale, flat);
  outs.reserve(G);
  int64_t at = 0;
  for (size_t g = 0; g < G; ++g) {
    const int64_t m = XQ[g].size(0), n = WQ[g].size(0);
    outs.push_back(flat.as_strided({m, n}, {n, 1}, at));
    at += m * n;
  }
  return outs;
}

Tensor grouped_cat_op(TensorList XQ, TensorList WQ, TensorList x_scale, TensorList w_scale) {
  check_grouped(XQ, WQ, x_scale, w_scale);
  TORCH_CHECK(XQ.size() > 0, "at least one group is required");
  const int64_t N = WQ[0].size(0);
  int64_t total = 0;
  for (size_t g = 0; g < XQ.size(); ++g) {
    TORCH_CHECK(WQ[g].size(0) == N, "all groups must share N to concatenate outputs");
    total += XQ[g].size(0);
  }
  Tensor Y = empty_on({total, N}, at::kBFloat16, XQ[0]);
  launch_grouped(XQ, WQ, x_scale, w_scale, Y);
  return Y;
}

// XQ [total_M, K], WQ [G, N, K], M_sizes int64 [G] on the GPU, never read on the host (fp8_rowwise_grouped_gemm.hip:607-655).
Tensor grouped_stacked_op(const Tensor& XQ, const Tensor& WQ, const Tensor& x_scale, const Tensor& w_scale, const Tensor& M_sizes) {
  TORCH_CHECK(XQ.is_cuda() && XQ.is_contiguous() && WQ.is_cuda() && WQ.is_contiguous(), "XQ/WQ must be contiguous GPU tensors");
  TORCH_CHECK(XQ.dim() == 2 && WQ.dim() == 3, "XQ must be 2-D [total_M, K] and WQ 3-D [G, N, K]");
  TORCH_CHECK(XQ.scalar_type() == kF8 && WQ.scalar_type() == kF8, "XQ and WQ must be torch.float8_e4m3fn on gfx950");
  TORCH_CHECK(x_scale.scalar_type() == at::kFloat && w_scale.scalar_type() == at::kFloat, "Scales must be float32.");
  TORCH_CHECK(M_sizes.is_cuda() && M_sizes.scalar_type() == at::kLong, "M_sizes must be an int64 GPU tensor");
  const int64_t total_M = XQ.size(0), K = XQ.size(1), G = WQ.size(0), N = WQ.size(1);
  TORCH_CHECK(K == WQ.size(2), "XQ and WQ must share K");
  TORCH_CHECK(M_sizes.numel() == G, "M_sizes must have one entry per group");
  TORCH_CHECK(x_scale.numel() == total_M && w_scale.numel() == G * N, "scale sizes must match total_M and G*N");
  TORCH_CHECK(WQ.device() == XQ.device() && x_scale.device() == XQ.device() && w_scale.device() == XQ.device() && M_sizes.device() == XQ.device(),
              "all operands must be on the same device");
  Tensor Y = empty_on({total_M, N}, at::kBFloat16, XQ);
  if (total_M == 0 || N == 0 || G == 0) return Y;
  if (K == 0) return Y.zero_();
  const auto xs = contiguous(x_scale), ws = contiguous(w_scale), ms = contiguous(M_sizes);
  const c10::DeviceGuard guard(XQ.device());
  check_rc(api.mslk_amd_f8f8bf16_rowwise_grouped_stacked(XQ.const_data_ptr(), WQ.const_data_ptr(), xs->const_data_ptr<float>(), ws->const_data_ptr<float>(),
                                                         ms->const_data_ptr<int64_t>(), (int)G, total_M, N, K, Y.mutable_data_ptr(), stream_of(XQ)));
  return Y;
}

// The torch._grouped_mm convention (fp8_rowwise_grouped_gemm.hip:720-845); the four layouts are listed in mslk_amd/gemm.py.
Tensor grouped_mm_op(const Tensor& XQ, const Tensor& WQ, const Tensor& x_scale, const Tensor& w_scale, const OptTensor& offsets, Tensor output) {
  TORCH_CHECK(XQ.is_cuda() && XQ.is_contiguous() && WQ.is_cuda() && WQ.is_contiguous(), "XQ/WQ must be contiguous GPU tensors");
  TORCH_CHECK(XQ.scalar_type() == WQ.scalar_type(), "XQ and WQ dtypes must match, got ", XQ.scalar_type(), " vs ", WQ.scalar_type());
  TORCH_CHECK(XQ.scalar_type() == kF8, "XQ and WQ must be torch.float8_e4m3fn on gfx950, got ", XQ.scalar_type());
  TORCH_CHECK(x_scale.scalar_type() == at::kFloat && w_scale.scalar_type() == at::kFloat, "Scales must be float32.");
  TORCH_CHECK(x_scale.is_contiguous() && w_scale.is_contiguous(), "scales must be contiguous");
  const bool has_offsets = offsets.has_value() && offsets->defined();
  auto need_offsets = [&](const char* what) {
    TORCH_CHECK(has_offsets, "Must pass offsets for 2D input ", what, ".");
    TORCH_CHECK(offsets->scalar_type() == at::kInt, "offsets must be int32.");
    TORCH_CHECK(offsets->is_cuda() && offsets->is_contiguous() && offsets->dim() == 1, "offsets must be a 1-D contiguous GPU tensor");
    return offsets->size(0);
  };
  auto shape_is = [](const Tensor& t, at::IntArrayRef s) { return t.sizes() == s; };
  int64_t G, M, N, K;
  int layout;
  if (XQ.dim() == 2 && WQ.dim() == 3) {
    G = need_offsets("XQ");
    M = XQ.size(0), N = WQ.size(1), K = WQ.size(2);
    layout = MSLK_AMD_GROUPS_M_OFFSETS;
    TORCH_CHECK(XQ.size(1) == K && WQ.size(0) == G, "XQ shape must be (total_M, K) and WQ shape must be (G, N, K).");
    TORCH_CHECK(x_scale.dim() >= 1 && x_scale.size(0) == M, "x_scale shape must be (total_M).");
    TORCH_CHECK(shape_is(w_scale, {G, N}), "w_scale shape must be (G, N).");
    TORCH_CHECK(shape_is(output, {M, N}), "out shape must be (total_M, N).");
  } else if (XQ.dim() == 3 && WQ.dim() == 2) {
    G = need_offsets("WQ");
    M = XQ.size(1), N = WQ.size(0), K = WQ.size(1);
    layout = MSLK_AMD_GROUPS_N_OFFSETS;
    TORCH_CHECK(XQ.size(0) == G && XQ.size(2) == K, "XQ shape must be (G, M, K) and WQ shape must be (total_N, K).");
    TORCH_CHECK(shape_is(x_scale, {G, M}), "x_scale shape must be (G, M).");
    TORCH_CHECK(w_scale.dim() >= 1 && w_scale.size(0) == N, "w_scale shape must be (total_N).");
    TORCH_CHECK(shape_is(output, {M, N}), "out shape must be (M, total_N).");
  } else if (XQ.dim() == 3 && WQ.dim() == 3) {
    TORCH_CHECK(!has_offsets, "Offsets should not be passed for 3D-3D inputs.");
    G = XQ.size(0), M = XQ.size(1), K = XQ.size(2), N = WQ.size(1);
    layout = MSLK_AMD_GROUPS_UNIFORM;
    TORCH_CHECK(WQ.size(0) == G && WQ.size(2) == K, "XQ shape must be (G, M, K) and WQ shape must be (G, N, K).");
    TORCH_CHECK(shape_is(x_scale, {G, M}), "x_scale shape must be (G, M).");
    TORCH_CHECK(shape_is(w_scale, {G, N}), "w_scale shape must be (G, N).");
    TORCH_CHECK(shape_is(output, {G, M, N}), "out shape must be (G, M, N).");
  } else if (XQ.dim() == 2 && WQ.dim() == 2) {
    G = need_offsets("s XQ and WQ");
    M = XQ.size(0), N = WQ.size(0), K = XQ.size(1);
    layout = MSLK_AMD_GROUPS_K_OFFSETS;
    TORCH_CHECK(WQ.size(1) == K, "XQ shape must be (M, total_K) and WQ shape must be (N, total_K).");
    TORCH_CHECK(x_scale.dim() >= 1 && x_scale.size(0) == G * M, "x_scale shape must be (G * M).");
    TORCH_CHECK(w_scale.dim() >= 1 && w_scale.size(0) == G * N, "w_scale shape must be (G * N).");
    TORCH_CHECK(shape_is(output, {G, M, N}), "out shape must be (G, M, N).");
  } else {
    TORCH_CHECK(false, "Invalid input shapes. Must be one of 2D-2D, 3D-3D, 2D-3D, 3D-2D.");
  }
  TORCH_CHECK(layout == MSLK_AMD_GROUPS_N_OFFSETS || N % 8 == 0, "N must be divisible by 8.");
  TORCH_CHECK(output.scalar_type() == at::kBFloat16 && output.is_cuda() && output.is_contiguous() && output.device() == XQ.device(),
              "output must be a contiguous bfloat16 GPU tensor on the device of XQ");
  TORCH_CHECK(WQ.device() == XQ.device() && x_scale.device() == XQ.device() && w_scale.device() == XQ.device() &&
                  (!has_offsets || offsets->device() == XQ.device()),
              "all operands must be on the same device");
  if (output.numel() == 0) return output;
  const c10::DeviceGuard guard(XQ.device());
  check_rc(api.mslk_amd_f8f8bf16_rowwise_grouped_mm(XQ.const_data_ptr(), WQ.const_data_ptr(), x_scale.const_data_ptr<float>(),
                                                    w_scale.const_data_ptr<float>(), has_offsets ? offsets->const_data_ptr<int32_t>() : nullptr,
                                                    layout, (int)G, M, N, K, output.mutable_data_ptr(), stream_of(XQ)));
  return output;
}

// Registered as boxed functions, one operator at a time and when the package asks for it.  A library loaded earlier may have
// defined an operator (the package then only replaces its GPU kernel): a kernel registered with its C++ type is refused where
// that library's own kernels take, say, Tensor by value instead of by reference, and an exception in a static initializer
// ends the process.  Calls from Python are boxed anyway.
template <auto FN>
void boxed(const c10::OperatorHandle& op, c10::DispatchKeySet keys, torch::jit::Stack* stack) {
  static const c10::KernelFunction kernel = c10::KernelFunction::makeFromUnboxedFunction(TORCH_FN(FN));
  kernel.callBoxed(op, keys, stack);
}
struct Kernel {
  const char *ns, *name;
  torch::CppFunction (*make)();
};
template <auto FN>
constexpr Kernel kernel(const char* ns, const char* name) {
  return {ns, name, [] { return torch::CppFunction::makeFromBoxedFunction<&boxed<FN>>(); }};
}
const Kernel kernels[] = {
    kernel<quantize_fp8_row>("triton", "quantize_fp8_row"),
    kernel<quantize_fp8_per_row>("mslk", "quantize_fp8_per_row"),
    kernel<dequantize_fp8_row>("mslk", "dequantize_fp8_row"),
    kernel<silu_mul_quant>("mslk", "silu_mul_quant"),
    kernel<gather_scale_quant_dense_tokens>("mslk", "gather_scale_quant_dense_tokens"),
    kernel<rowwise_op<false, false>>("mslk", "f8f8bf16_rowwise"),
    kernel<rowwise_op<true, false>>("mslk", "f8f8f16_rowwise"),
    kernel<rowwise_op<false, true>>("mslk", "f8f8bf16_rowwise_preshuffle"),
    kernel<rowwise_op<true, true>>("mslk", "f8f8f16_rowwise_preshuffle"),
    kernel<rowwise_out_op>("mslk", "f8f8bf16_rowwise_out"),
    kernel<quantize_rowwise>("mslk", "quantize_f8f8bf16_rowwise"),
    kernel<grouped_op>("mslk", "f8f8bf16_rowwise_grouped"),
    kernel<grouped_cat_op>("mslk", "f8f8bf16_rowwise_grouped_cat"),
    kernel<grouped_stacked_op>("mslk", "f8f8bf16_rowwise_grouped_stacked"),
    kernel<grouped_mm_op>("mslk", "f8f8bf16_rowwise_grouped_mm"),
};

}  // namespace

// Binds the entry points of the library at `path`, all of them or none; returns an error message or null.
extern "C" const char* mslk_amd_torch_bind(const char* path) {
  void* lib = dlopen(path, RTLD_NOW | RTLD_LOCAL);
  if (lib == nullptr) return dlerror();
  Api bound;
#define X(name)                                                                              \
  bound.name = reinterpret_cast<decltype(bound.name)>(dlsym(lib, #name));                      \
  if (bound.name == nullptr) {                                                                 \
    dlclose(lib);                                                                              \
    return "the library does not export " #name;                                               \
  }
  MSLK_AMD_ENTRY_POINTS(X)
#undef X
  api = bound;
  return nullptr;
}

// Makes the native function the GPU kernel of operator `name` in namespace `ns`, whose schema has to have the types of the
// one the package defines; after mslk_amd_torch_bind().  Returns an error message or null.
extern "C" const char* mslk_amd_torch_register(const char* ns, const char* name) {
  static std::string error;   // calls come from the import of the package, one at a time
  if (api.mslk_amd_last_error == nullptr) return "mslk_amd_torch_bind() comes first";
  for (const Kernel& k : kernels) {
    if (std::strcmp(k.ns, ns) != 0 || std::strcmp(k.name, name) != 0) continue;
    try {
      // kept until the process ends: the registration goes with the object
      auto* library = new torch::Library(torch::Library::IMPL, ns, c10::DispatchKey::CUDA, __FILE__, __LINE__);
      library->impl(name, k.make());
      return nullptr;
    } catch (const std::exception& e) {
      error = e.what();
      return error.c_str();
    }
  }
  return "no native kernel of this name";
}
