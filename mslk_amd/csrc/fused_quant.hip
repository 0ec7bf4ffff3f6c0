// Fused producers of the quantized MoE activations for gfx950: the row is produced in fp32
// (SiLU-gated product, or a gathered token times its routing score) and quantized to e4m3fn in the
// same pass, so the fp32 / bf16 intermediate never goes to HBM.
//
//   silu_mul_quant                  (reference: _mslk_silu_mul_quant, mslk/moe/activation.py:232-300)
//       y = x0 * sigmoid(x0) * x1                       fp32, evaluated left to right
//   gather_scale_quant_dense_tokens (reference: _mslk_gather_scale_fp8_rowwise_quant_dense_tokens,
//                                    mslk/moe/gather_scatter.py:545-640)
//       y = x[token[i]] * scores[token[i], expert[i]]   fp32
// followed in both by the quantization of those kernels:
//   row_max = clamp(max|y|, 1e-12 [, *scale_ub]);  s = 448 / row_max;  out_scale = 1 / s;
//   code = e4m3fn_rne(clamp(y * s, -448, 448))
// (saturating, unlike the stand-alone quantizer whose contract is the reference's torch branch).
// The two divisions of the scale are IEEE-correct; sigmoid is rcp(1 + exp(-x)) on the hardware
// transcendental units, accurate to a few fp32 ulp.
//
// HBM-bound (silu: 4 B in + 1 B out per element for 16-bit inputs; gather: 2 B in + 1 B out).  A wavefront or a
// workgroup owns a row; the produced fp32 values stay in registers between the
// maximum pass and the convert pass for rows of up to 16384 elements.
#include "common.h"
#include "kernels.h"
#include "rows.h"

namespace mslk_amd {
namespace {

constexpr float kMaxFp8 = 448.0f;
constexpr float kEps = 1e-12f;

template <int DTYPE>
MSLK_AMD_DEVINL float elem_to_f32(uint32_t bits) {
  if constexpr (DTYPE == 0) return bf16_bits_to_f32(bits);
  else return (float)__builtin_bit_cast(_Float16, (unsigned short)bits);
}

MSLK_AMD_DEVINL float load_scalar_f32(const void* p, int64_t idx, int dtype) {
  if (dtype == 2) return static_cast<const float*>(p)[idx];
  const uint32_t b = static_cast<const uint16_t*>(p)[idx];
  return dtype == 0 ? bf16_bits_to_f32(b) : (float)__builtin_bit_cast(_Float16, (unsigned short)b);
}

MSLK_AMD_DEVINL int64_t load_index(const void* p, int64_t i, int is_i64) {
  return is_i64 ? static_cast<const int64_t*>(p)[i] : (int64_t) static_cast<const int32_t*>(p)[i];
}

// exp(-a) through the hardware base-2 exponential (1 ulp); the rounding error of the product
// -a * log2(e) is carried separately and folded back in, so the result stays within about 2 ulp for
// every argument instead of growing with |a|.
MSLK_AMD_DEVINL float exp_neg(float a) {
  constexpr float kLog2eHi = 1.44269502162933349609375f, kLog2eLo = 1.925963033500011e-8f, kLn2 = 0.693147182464599609375f;
  const float na = -a;
  const float t = na * kLog2eHi;
  float e = __builtin_fmaf(na, kLog2eHi, -t);
  e = __builtin_fmaf(na, kLog2eLo, e);
  const float p = __builtin_amdgcn_exp2f(t);
  return __builtin_fmaf(p, e * kLn2, p);
}

// sigmoid through the hardware reciprocal (1 ulp): the convert that follows keeps 3 mantissa bits.
MSLK_AMD_DEVINL float silu_mul(float a, float b) {
  const float sig = __builtin_amdgcn_rcpf(1.0f + exp_neg(a));
  return (a * sig) * b;
}

// 8 consecutive 16-bit elements -> fp32
template <int DTYPE>
MSLK_AMD_DEVINL void unpack8(const v4u& w, float (&f)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = elem_to_f32<DTYPE>(w[i] & 0xFFFFu);
    f[2 * i + 1] = elem_to_f32<DTYPE>(w[i] >> 16);
  }
}

// The row a workgroup works on, resolved once per workgroup.
struct RowSource {
  const char* a;    // x0 row, or the gathered x row
  const char* b;    // x1 row (silu only)
  float score;      // gather only
  bool live;
};

template <int OP>
MSLK_AMD_DEVINL RowSource resolve_row(const FusedQuantArgs& p, int64_t row) {
  RowSource r{nullptr, nullptr, 1.0f, false};
  if (p.valid_count != nullptr && row >= load_index(p.valid_count, 0, p.valid_is_i64)) return r;
  if constexpr (OP == kFusedSiluMul) {
    r.a = static_cast<const char*>(p.x0) + row * p.stride0 * 2;
    r.b = static_cast<const char*>(p.x1) + row * p.stride1 * 2;
    r.live = true;
  } else {
    const int64_t t = load_index(p.token_idx, row, p.token_is_i64);
    const int64_t e = load_index(p.expert_idx, row, p.expert_is_i64);
    if (t < 0 || t >= p.T || e < 0 || e >= p.E) return r;   // an index outside the tensors: touch nothing
    r.a = static_cast<const char*>(p.x0) + t * p.stride0 * 2;
    r.score = load_scalar_f32(p.scores, t * p.stride_t + e * p.stride_e, p.score_dtype);
    r.live = true;
  }
  return r;
}

// Eight elements of the row from its 16 input bytes (32 for the gated product).
template <int OP, int DTYPE>
MSLK_AMD_DEVINL void produce8(const v4u& va, const v4u& vb, float score, float (&y)[8]) {
  float a[8];
  unpack8<DTYPE>(va, a);
  if constexpr (OP == kFusedSiluMul) {
    float b[8];
    unpack8<DTYPE>(vb, b);
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = silu_mul(a[i], b[i]);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = a[i] * score;
  }
}
template <int OP, int DTYPE>
MSLK_AMD_DEVINL void produce8(const RowSource& r, int vec, float (&y)[8]) {
  const v4u va = __builtin_nontemporal_load(reinterpret_cast<const v4u*>(r.a) + vec);
  v4u vb = va;
  if constexpr (OP == kFusedSiluMul) vb = __builtin_nontemporal_load(reinterpret_cast<const v4u*>(r.b) + vec);
  produce8<OP, DTYPE>(va, vb, r.score, y);
}

template <int OP, int DTYPE>
MSLK_AMD_DEVINL float produce1(const FusedQuantArgs& p, const RowSource& r, int k) {
  const float a = elem_to_f32<DTYPE>(reinterpret_cast<const uint16_t*>(r.a)[k]);
  if constexpr (OP == kFusedSiluMul) return silu_mul(a, elem_to_f32<DTYPE>(reinterpret_cast<const uint16_t*>(r.b)[k]));
  else return a * r.score;
}

// |y| as raw bits orders like the value for non-negative floats and puts every NaN above +inf.
MSLK_AMD_DEVINL void row_scales(uint32_t max_bits, const float* scale_ub, float& s, float& inv) {
  const float amax = __uint_as_float(max_bits);
  float c = (amax < kEps) ? kEps : amax;
  if (scale_ub != nullptr) c = (c > *scale_ub) ? *scale_ub : c;
  s = kMaxFp8 / c;
  inv = 1.0f / s;
}

MSLK_AMD_DEVINL v2u quantize8_saturating(const float (&y)[8], float s) {
  float f[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) f[i] = __builtin_amdgcn_fmed3f(y[i] * s, -kMaxFp8, kMaxFp8);   // clamp; a NaN comes out as -448, as from fmin(fmax())
  // within +-448 the hardware conversion alone gives the codes (no NaN / overflow fix-up to apply)
  v2u r;
  r.x = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], __builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], 0, false), true);
  r.y = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(f[6], f[7], __builtin_amdgcn_cvt_pk_fp8_f32(f[4], f[5], 0, false), true);
  return r;
}

// Vector path: D % 8 == 0, input rows 16-byte aligned, output rows 8-byte aligned, at most TEAM * NV vectors of eight per
// row, whose produced values stay in registers.  Bound by HBM: all loads of a lane are in flight before the first value is
// formed (rows.h).  Against loads that waited for each other, bf16: gather 8192 x 5120 27.4 -> 21.8 us (5.8 TB/s), 32768 x 2048
// 39.1 -> 33.1 (6.1 TB/s), 16384 x 1408 16.2 -> 13.6; the gated product, which had two loads per vector in flight, 8192 x
// 4096 27.4 -> 27.1 (6.2 TB/s), 32768 x 2048 53.7 -> 49.6 (6.8 TB/s).
// TEAM = 64: one wavefront per row, four rows per workgroup (rows of MoE intermediate sizes in large numbers); otherwise
// one workgroup of TEAM lanes per row.
template <int OP, int DTYPE, int TEAM, int NV>
__global__ __launch_bounds__(256) void fused_quant_vec_kernel(FusedQuantArgs p) {
  static_assert(TEAM == kWave || TEAM == 256, "a wavefront or a workgroup of four per row");
  __shared__ uint32_t smem[4];
  const int64_t row = TEAM == kWave ? (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : row_block();
  if (row >= p.rows) return;                     // uniform over the team, the wavefront or (with the barrier) the workgroup
  const RowSource r = resolve_row<OP>(p, row);   // uniform over the team
  if (!r.live) return;
  const int lane = threadIdx.x % TEAM;
  const buffer_t src_a = make_buffer(r.a, (uint32_t)p.D * 2);
  const buffer_t src_b = make_buffer(OP == kFusedSiluMul ? r.b : r.a, (uint32_t)p.D * 2);
  v4u va[NV], vb[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    va[i] = buffer_load16(src_a, (uint32_t)(i * TEAM + lane) * 16);
    if constexpr (OP == kFusedSiluMul) vb[i] = buffer_load16(src_b, (uint32_t)(i * TEAM + lane) * 16);
  }
  // Whether the wavefront owns any part of vector i.  One wholly beyond the row reads as zero and is not worth the arithmetic of
  // the gated product (131072 x 2056: 286 -> 227 us, 2047 x 8200: 18.9 -> 14.0).  (The empty instruction keeps the loads where
  // they are: the compiler would move each into the branch that uses it, one round trip each; and the wait is there for the
  // loads of the branches not taken, before their registers are used again -- the compiler would put it between the stores.)
  constexpr bool SKIP = OP == kFusedSiluMul && TEAM > kWave && NV > 1;
  const int wave_first = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * kWave;
  auto used = [&](int i) { return !SKIP || i * TEAM + wave_first < p.D >> 3; };
  if constexpr (SKIP) asm volatile("" : : : "memory");
  float y[NV][8];
  uint32_t m = 0;
#pragma unroll
  for (int i = 0; i < NV; ++i) {   // lanes beyond the row read as zero and produce zero
    if (!used(i)) break;
    produce8<OP, DTYPE>(va[i], vb[i], r.score, y[i]);
#pragma unroll
    for (int e = 0; e < 8; ++e) m = max(m, __float_as_uint(y[i][e]) & 0x7FFFFFFFu);
  }
  if constexpr (OP == kFusedGatherScale) {
    // (0 * score is NaN for an infinite or NaN score: a vector beyond the row must not enter the maximum then)
    if (!(__builtin_fabsf(r.score) < __builtin_inff())) {
      m = 0;
#pragma unroll
      for (int i = 0; i < NV; ++i)
        if (i * TEAM + lane < (p.D >> 3))
#pragma unroll
          for (int e = 0; e < 8; ++e) m = max(m, __float_as_uint(y[i][e]) & 0x7FFFFFFFu);
    }
  }
  if constexpr (SKIP) __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
  m = team_max<TEAM>(m, smem);
  float s, inv;
  row_scales(m, p.scale_ub, s, inv);
  if (lane == 0) p.out_scale[row] = inv;
  const buffer_t dst = make_buffer(p.out + row * (int64_t)p.D, (uint32_t)p.D);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    if (!used(i)) break;
    buffer_store8_through(dst, (uint32_t)(i * TEAM + lane) * 8, quantize8_saturating(y[i], s));
  }
}

// Rows of any length: as above, produced twice.
template <int OP, int DTYPE>
__global__ __launch_bounds__(256) void fused_quant_long_kernel(FusedQuantArgs p) {
  __shared__ uint32_t smem[4];
  const int64_t row = blockIdx.x;
  const RowSource r = resolve_row<OP>(p, row);
  if (!r.live) return;
  const int nvec = p.D >> 3;
  uint32_t m = 0;
  float y[8];
  for (int vec = threadIdx.x; vec < nvec; vec += 256) {
    produce8<OP, DTYPE>(r, vec, y);
#pragma unroll
    for (int e = 0; e < 8; ++e) m = max(m, __float_as_uint(y[e]) & 0x7FFFFFFFu);
  }
  m = team_max<256>(m, smem);
  float s, inv;
  row_scales(m, p.scale_ub, s, inv);
  if (threadIdx.x == 0) p.out_scale[row] = inv;
  uint8_t* out_row = p.out + row * (int64_t)p.D;
  for (int vec = threadIdx.x; vec < nvec; vec += 256) {
    produce8<OP, DTYPE>(r, vec, y);
    const v2u q = quantize8_saturating(y, s);
    store8_write_through(out_row + (int64_t)vec * 8, v2i{(int)q.x, (int)q.y});
  }
}

// Any D, any alignment: scalar accesses, the row is produced twice.
template <int OP, int DTYPE>
__global__ __launch_bounds__(256) void fused_quant_generic_kernel(FusedQuantArgs p) {
  __shared__ uint32_t smem[4];
  const int64_t row = blockIdx.x;
  const RowSource r = resolve_row<OP>(p, row);
  if (!r.live) return;
  uint32_t m = 0;
  for (int k = threadIdx.x; k < p.D; k += 256) m = max(m, __float_as_uint(produce1<OP, DTYPE>(p, r, k)) & 0x7FFFFFFFu);
  m = team_max<256>(m, smem);
  float s, inv;
  row_scales(m, p.scale_ub, s, inv);
  if (threadIdx.x == 0) p.out_scale[row] = inv;
  for (int k = threadIdx.x; k < p.D; k += 256) {
    const float f = __builtin_fminf(__builtin_fmaxf(produce1<OP, DTYPE>(p, r, k) * s, -kMaxFp8), kMaxFp8);
    p.out[row * (int64_t)p.D + k] = (uint8_t)(cvt_pk_e4m3fn(f, 0.0f) & 0xFFu);
  }
}

template <int OP, int DTYPE>
hipError_t launch_fused_t(const FusedQuantArgs& p, hipStream_t s) {
  const unsigned rows = (unsigned)p.rows;
  const bool vec_ok = p.D % 8 == 0 && reinterpret_cast<uintptr_t>(p.x0) % 16 == 0 && (p.stride0 * 2) % 16 == 0 &&
                      (OP != kFusedSiluMul || (reinterpret_cast<uintptr_t>(p.x1) % 16 == 0 && (p.stride1 * 2) % 16 == 0)) &&
                      reinterpret_cast<uintptr_t>(p.out) % 8 == 0;
  if (!vec_ok) {
    fused_quant_generic_kernel<OP, DTYPE><<<rows, 256, 0, s>>>(p);
    return hipGetLastError();
  }
  auto team = [&](auto t, auto n) {
    constexpr int TEAM = decltype(t)::value, NV = decltype(n)::value;
    fused_quant_vec_kernel<OP, DTYPE, TEAM, NV><<<TEAM == kWave ? dim3((rows + 3) / 4) : row_grid(p.rows), 256, 0, s>>>(p);
    return hipGetLastError();
  };
  // As few vectors as hold the row: one beyond its end costs the arithmetic all the same (32768 x 768, gated product: 64 x 2
  // 22.2, 64 x 4 35.1 us).  In large numbers short rows take a wavefront each (gather, 32768 x 2048: 64 x 4 33.1, 256 45.1).
  // The gated product computes more per byte, so that lanes without a vector cost it more: a wavefront for up to two vectors
  // whatever the number of rows (2047 x 512 fp16: 3.9, as 256 x 1 4.7), in large numbers for up to three (131072 x 1408
  // fp16: 139, as 256 x 1 171), but not for four (32768 x 2048: 256 49.6, 64 x 4 52.3).
  if (OP == kFusedSiluMul ? p.D <= 1024 || (p.rows >= 2048 && p.D <= 1536) : p.rows >= 2048 && p.D <= 2048) {
    if (p.D <= 512) return team(Int<64>{}, Int<1>{});
    if (p.D <= 1024) return team(Int<64>{}, Int<2>{});
    return team(Int<64>{}, Int<(OP == kFusedSiluMul ? 3 : 4)>{});
  }
  if (p.D <= 2048) return team(Int<256>{}, Int<1>{});
  if (p.D <= 4096) return team(Int<256>{}, Int<2>{});
  if (p.D <= 6144) return team(Int<256>{}, Int<3>{});
  if (p.D <= 8192) return team(Int<256>{}, Int<4>{});
  if (p.D <= 16384) return team(Int<256>{}, Int<8>{});
  fused_quant_long_kernel<OP, DTYPE><<<rows, 256, 0, s>>>(p);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_fused_quant(const FusedQuantArgs& p, int op, hipStream_t s) {
  if (p.rows <= 0 || p.D <= 0) return hipSuccess;
  if (op == kFusedSiluMul) return p.dtype == 0 ? launch_fused_t<kFusedSiluMul, 0>(p, s) : launch_fused_t<kFusedSiluMul, 1>(p, s);
  if (op == kFusedGatherScale)
    return p.dtype == 0 ? launch_fused_t<kFusedGatherScale, 0>(p, s) : launch_fused_t<kFusedGatherScale, 1>(p, s);
  return hipErrorInvalidValue;
}

}  // namespace mslk_amd
