// Row-wise FP8 (e4m3fn) quantizer for gfx950.
//
// Bit-exact to the torch branch of the reference's quantize_fp8_row
// (mslk/quantize/triton/fp8_quantize.py:360-378):
//   amax  = max|x| over the row, taken in the input dtype (exact for bf16/fp16/fp32)
//   amax  = clamp(amax, min = dtype(1e-12) [, max = dtype(*scale_ub)]), NaN propagates
//   inv   = fl32(fl32(1 / amax) * 448);  inv == +inf -> 1
//   code  = e4m3fn_rne(fl32(fl32(x) * inv))            (no saturation: > 464 becomes NaN)
//   scale = fl32(1 / inv)
//
// TRITON = true selects the arithmetic of the reference's GPU (Triton) kernel instead
// (mslk/quantize/triton/fp8_quantize.py:131-207): amax clamped at `eps` (default 1/512) [and *scale_ub],
//   scale = fl32(amax / 448);  code = e4m3fn_rne(clamp(fl32(fl32(x) / scale), -448, 448))
// with IEEE-correct divisions (div_rn) and saturation.
//
// The pass is HBM-bound (2 B in + 1 B out per element for bf16), so the kernel is organised
// around 128-bit coalesced loads that stay in registers between the amax pass and the convert
// pass: a row is owned by a "team" of 8 ... 1024 lanes, each of which keeps NV vectors of 8 elements.
// Rows beyond that are streamed twice (the second read hits L2 / Infinity Cache).
#include "common.h"
#include "kernels.h"
#include "quant_math.h"
#include "rows.h"

namespace mslk_amd {
namespace {

// 8 consecutive elements of a row.
template <int DTYPE> struct Vec8 { v4u w; };            // 8 x 16-bit
template <> struct Vec8<2> { v4u lo, hi; };             // 8 x fp32

template <int DTYPE>
MSLK_AMD_DEVINL Vec8<DTYPE> load_vec8(buffer_t row, uint32_t off) {
  Vec8<DTYPE> v;
  if constexpr (DTYPE == 2) {
    v.lo = buffer_load16(row, off);
    v.hi = buffer_load16(row, off + 16);
  } else {
    v.w = buffer_load16(row, off);
  }
  return v;
}

// Rows longer than the registers hold: 64-bit addressing, streamed twice.
template <int DTYPE>
MSLK_AMD_DEVINL Vec8<DTYPE> load_vec8(const void* row_ptr, int vec_idx) {
  Vec8<DTYPE> v;
  if constexpr (DTYPE == 2) {
    const v4u* p = reinterpret_cast<const v4u*>(row_ptr) + 2 * (int64_t)vec_idx;
    v.lo = __builtin_nontemporal_load(p);
    v.hi = __builtin_nontemporal_load(p + 1);
  } else {
    v.w = __builtin_nontemporal_load(reinterpret_cast<const v4u*>(row_ptr) + vec_idx);
  }
  return v;
}

// Running maximum of |x| kept as raw bits: for non-negative IEEE values unsigned integer order
// equals numeric order and every NaN pattern sorts above +inf, so a NaN in the row survives.
template <int DTYPE>
MSLK_AMD_DEVINL uint32_t absmax_bits(uint32_t m, const Vec8<DTYPE>& v) {
  if constexpr (DTYPE == 2) {
#pragma unroll
    for (int i = 0; i < 4; ++i) m = max(max(m, v.lo[i] & 0x7FFFFFFFu), v.hi[i] & 0x7FFFFFFFu);
    return m;
  } else {
    us2 acc = __builtin_bit_cast(us2, m);
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_elementwise_max(acc, __builtin_bit_cast(us2, v.w[i] & 0x7FFF7FFFu));
    return __builtin_bit_cast(uint32_t, acc);
  }
}

template <int DTYPE>
MSLK_AMD_DEVINL uint32_t finish_absmax_bits(uint32_t m) {
  if constexpr (DTYPE == 2) return m;
  return max(m & 0xFFFFu, m >> 16);
}

// clamp(v, -448, 448) in one instruction (the median of the three; a NaN comes out as -448, like fmin(fmax(v, -448), 448))
MSLK_AMD_DEVINL float clamp448(float v) { return __builtin_amdgcn_fmed3f(v, -448.0f, 448.0f); }

// Four fp32 within +-464 -> four codes by the hardware conversion alone.
MSLK_AMD_DEVINL uint32_t cvt4_plain(float a, float b, float c, float d) {
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(c, d, __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false), true);
}

// How a row's elements become codes; the same for the whole row.
enum RowMode : int {
  kModePlain = 0,    // a finite row maximum that scale_ub has not cut: no quotient exceeds 448 (1 + 2^-22), the bare
                     // conversion gives the codes.  Torch arithmetic: x * factor.  Triton arithmetic: x / factor with a
                     // reciprocal and two FMAs, q0 = x r, e = fma(q0, factor, -x), q = fma(-e, r, q0) with r =
                     // fl32(1 / factor).  The codes are those of the IEEE division for every 16-bit element under every
                     // 16-bit row maximum of at least 2^-64 (exhaustively checked on the CPU, tests/test_oracle.py; an
                     // exact quotient leaves e = +0, and -0 added to q0 keeps the sign of a zero).
  kModeGeneral = 1,  // torch arithmetic with the NaN / overflow fix-up; Triton arithmetic with IEEE divisions and the clamp
};
template <int DTYPE, bool TRITON, int MODE>
MSLK_AMD_DEVINL v2u quantize_vec8(const Vec8<DTYPE>& v, float factor, float rcp) {
  float f[8];
  if constexpr (DTYPE == 2) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f[i] = __uint_as_float(v.lo[i]);
      f[4 + i] = __uint_as_float(v.hi[i]);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f[2 * i] = Traits<DTYPE>::to_f32(v.w[i] & 0xFFFFu);
      f[2 * i + 1] = Traits<DTYPE>::to_f32(v.w[i] >> 16);
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    if constexpr (!TRITON) {
      f[i] = f[i] * factor;
    } else if constexpr (MODE == kModePlain) {
      const float q0 = f[i] * rcp;
      f[i] = __builtin_fmaf(-__builtin_fmaf(q0, factor, -f[i]), rcp, q0);
    } else {
      f[i] = clamp448(f[i] / factor);   // within +-448, so the bare conversion serves here too
    }
  }
  if constexpr (TRITON || MODE == kModePlain) {
    return v2u{cvt4_plain(f[0], f[1], f[2], f[3]), cvt4_plain(f[4], f[5], f[6], f[7])};
  } else {
    return v2u{cvt_pk_e4m3fn(f[0], f[1]) | (cvt_pk_e4m3fn(f[2], f[3]) << 16),
               cvt_pk_e4m3fn(f[4], f[5]) | (cvt_pk_e4m3fn(f[6], f[7]) << 16)};
  }
}

// Jagged rows (reference: JAGGED branch of _kernel_quantize_fp8_row, fp8_quantize.py:123-129): rows are
// grouped in blocks of `rows_per_group`; inside block b only the first zero_start[b] rows hold data,
// the others are treated as all-zero rows and are never read.
struct JaggedRows {
  const void* zero_start;   // nullptr: every row is live
  int64_t rows_per_group;
  int index_is_i32;
  float triton_eps;         // lower bound of amax in the TRITON arithmetic
};

MSLK_AMD_DEVINL bool row_is_live(const JaggedRows& j, int64_t row) {
  if (j.zero_start == nullptr) return true;
  const int64_t b = row / j.rows_per_group, n = row - b * j.rows_per_group;
  const int64_t live = j.index_is_i32 ? (int64_t) static_cast<const int32_t*>(j.zero_start)[b]
                                      : static_cast<const int64_t*>(j.zero_start)[b];
  return n < live;
}

// Whether a row takes kModePlain; in the Triton arithmetic `rcp` is then the reciprocal of the divisor.
template <int DTYPE, bool TRITON>
MSLK_AMD_DEVINL bool row_is_plain(float amax, const float* scale_ub, float triton_eps, float divisor, float& rcp) {
  rcp = 0.f;
  if (scale_ub != nullptr || !(amax < __builtin_inff())) return false;
  if constexpr (!TRITON) return true;
  if constexpr (DTYPE == 2) return false;   // fp32 elements: the short division is proven for 16-bit ones only
  if (!(amax >= triton_eps && amax >= 0x1p-64f)) return false;
  rcp = 1.0f / divisor;
  return true;
}

// Vector path: K % 8 == 0, row starts 16-byte aligned, output rows 8-byte aligned, at most TEAM * NV vectors of eight
// elements per row.  TEAM lanes own a row: several rows per wavefront (TEAM < 64), one per wavefront, or one per
// workgroup of TEAM >= 256 lanes.  Bound by HBM: all NV loads of a lane are in flight before the maximum is formed
// (rows.h).  Against loads that waited for each other, Triton arithmetic on bf16: 4096 x 4096 11.9 -> 10.0 us (5.0 TB/s),
// 8192 x 8192 41.8 -> 30.5 (6.6 TB/s), 131072 x 128 16.7 -> 10.8, 64 x 14336 4.9 -> 3.4 (the cost of a launch).
// PART: a vector wholly beyond the row of a wavefront reads as zero, but is not worth its arithmetic (1024 x 16392 with scale_ub,
// Triton arithmetic: 17.5 -> 12.9 us; 2047 x 64, three of four wavefronts without a vector: 4.3 -> 3.8).  A kernel of its own:
// the branches between the vectors keep their conversions apart (40 ns).
template <int DTYPE, int TEAM, int NV, bool TRITON, bool PART>
__global__ __launch_bounds__(TEAM > 256 ? TEAM : 256) void quantize_rows_vec_kernel(
    const void* __restrict__ x, int64_t rows, int K, int64_t in_stride, uint8_t* __restrict__ out,
    int64_t out_stride, float* __restrict__ scale, const float* __restrict__ scale_ub, JaggedRows jag) {
  constexpr int BLOCK = TEAM > 256 ? TEAM : 256, TEAMS = BLOCK / TEAM;
  constexpr int ELEM_BYTES = (DTYPE == 2) ? 4 : 2;
  constexpr int ROWS_W = TEAM < kWave ? kWave / TEAM : 1;   // rows of a wavefront
  static_assert(TEAM <= kWave || TEAM == BLOCK, "a team is part of a wavefront, a wavefront or the workgroup");
  __shared__ uint32_t smem[BLOCK / kWave];
  const int lane = threadIdx.x % TEAM;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t row0 = (TEAM <= kWave ? (int64_t)blockIdx.x : row_block()) * TEAMS + (TEAM <= kWave ? wave * ROWS_W : 0);   // first row of the wavefront
  const int sub = TEAM < kWave ? (threadIdx.x & 63) / TEAM : 0;
  const int64_t row = row0 + sub;
  const bool valid = row < rows;
  const bool live = valid && row_is_live(jag, row);   // the same in every lane of the team
  const int64_t base_row = row0 < rows ? row0 : 0;
  const uint32_t nvec = (uint32_t)K >> 3;
  // one row per descriptor, whose size ends the row; several rows per descriptor when the team is part of a wavefront
  const buffer_t src = make_buffer(static_cast<const char*>(x) + base_row * in_stride * ELEM_BYTES,
                                   TEAM < kWave ? 0x7FFFFFF0u : (live ? (uint32_t)K * ELEM_BYTES : 0u));
  const buffer_t dst = make_buffer(out + base_row * out_stride, TEAM < kWave ? 0x7FFFFFF0u : (valid ? (uint32_t)K : 0u));
  auto at = [&](int i, bool ok, uint32_t stride, uint32_t vec_bytes) {   // byte offset of vector i of this lane
    const uint32_t v = i * TEAM + lane;
    if constexpr (TEAM < kWave) return ok && v < nvec ? sub * stride + v * vec_bytes : kBeyondBuffer;
    return v * vec_bytes;
  };
  auto pad = [&] {   // zero padding columns [K, out_stride)
    if (valid)
      for (int64_t k = K + lane; k < out_stride; k += TEAM) out[row * out_stride + k] = 0;
  };
  Vec8<DTYPE> cache[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) cache[i] = load_vec8<DTYPE>(src, at(i, live, (uint32_t)in_stride * ELEM_BYTES, 8 * ELEM_BYTES));
  // A wavefront without a live row (where rows are as wide as a workgroup, the whole workgroup): zero codes, whatever scale_ub
  // makes of the scale (0 / 0 is no zero), and nothing reduced.  (Behind the loads, which read no memory there: 40 ns less for
  // every other row.)
  if (jag.zero_start != nullptr && __ballot(live) == 0) {
    float inv, sc;
    scales_from_amax<DTYPE, TRITON>(0.f, scale_ub, jag.triton_eps, inv, sc);
    if (lane == 0 && valid) scale[row] = sc;
#pragma unroll
    for (int i = 0; i < NV; ++i) buffer_store8_through(dst, at(i, valid, (uint32_t)out_stride, 8), v2u{0, 0});
    pad();
    return;
  }
  uint32_t m = 0;
#pragma unroll
  for (int i = 0; i < NV; ++i) m = absmax_bits<DTYPE>(m, cache[i]);   // vectors beyond the row and dead rows read as zero
  m = team_max<TEAM>(finish_absmax_bits<DTYPE>(m), smem);

  // Whether the wavefront owns any part of vector i (PART: some wavefront does not).
  auto used = [&](int i) { return !PART || (uint32_t)(i * TEAM + (TEAM > kWave ? wave * kWave : 0)) < nvec; };
  float inv, sc, rcp;
  const float amax = Traits<DTYPE>::abs_bits_to_f32(m);
  scales_from_amax<DTYPE, TRITON>(amax, scale_ub, jag.triton_eps, inv, sc);
  if (lane == 0 && valid) scale[row] = sc;
  if (row_is_plain<DTYPE, TRITON>(amax, scale_ub, jag.triton_eps, inv, rcp)) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      if (!used(i)) break;
      buffer_store8_through(dst, at(i, valid, (uint32_t)out_stride, 8), quantize_vec8<DTYPE, TRITON, kModePlain>(cache[i], inv, rcp));
    }
  } else {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      if (!used(i)) break;
      v2u q = quantize_vec8<DTYPE, TRITON, kModeGeneral>(cache[i], inv, rcp);
      if (TEAM < kWave && !live) q = v2u{0, 0};   // a dead row beside live ones of the wavefront
      buffer_store8_through(dst, at(i, valid, (uint32_t)out_stride, 8), q);
    }
  }
  pad();
}

// Vector path for rows beyond the registers: one workgroup per row, read twice (the second read hits the caches).
template <int DTYPE, bool TRITON>
__global__ __launch_bounds__(256) void quantize_rows_long_kernel(
    const void* __restrict__ x, int64_t rows, int K, int64_t in_stride, uint8_t* __restrict__ out,
    int64_t out_stride, float* __restrict__ scale, const float* __restrict__ scale_ub, JaggedRows jag) {
  constexpr int ELEM_BYTES = (DTYPE == 2) ? 4 : 2;
  __shared__ uint32_t smem[4];
  const int64_t row = blockIdx.x;
  const int nvec = row_is_live(jag, row) ? K >> 3 : 0;
  const char* row_ptr = reinterpret_cast<const char*>(x) + row * in_stride * ELEM_BYTES;
  uint32_t m = 0;
  for (int idx = threadIdx.x; idx < nvec; idx += 256) m = absmax_bits<DTYPE>(m, load_vec8<DTYPE>(row_ptr, idx));
  m = team_max<256>(finish_absmax_bits<DTYPE>(m), smem);
  float inv, sc, rcp;
  const float amax = Traits<DTYPE>::abs_bits_to_f32(m);
  scales_from_amax<DTYPE, TRITON>(amax, scale_ub, jag.triton_eps, inv, sc);
  if (threadIdx.x == 0) scale[row] = sc;
  uint8_t* out_row = out + row * out_stride;
  if (row_is_plain<DTYPE, TRITON>(amax, scale_ub, jag.triton_eps, inv, rcp)) {
    for (int idx = threadIdx.x; idx < nvec; idx += 256) {
      const v2u q = quantize_vec8<DTYPE, TRITON, kModePlain>(load_vec8<DTYPE>(row_ptr, idx), inv, rcp);
      store8_write_through(out_row + (int64_t)idx * 8, v2i{(int)q.x, (int)q.y});
    }
  } else {
    for (int idx = threadIdx.x; idx < nvec; idx += 256) {
      const v2u q = quantize_vec8<DTYPE, TRITON, kModeGeneral>(load_vec8<DTYPE>(row_ptr, idx), inv, rcp);
      store8_write_through(out_row + (int64_t)idx * 8, v2i{(int)q.x, (int)q.y});
    }
  }
  // padding columns, and all of a dead row (out_stride and the row's start are multiples of 8)
  for (int64_t k = (int64_t)nvec * 8 + threadIdx.x * 8; k < out_stride; k += 256 * 8) store8_write_through(out_row + k, v2i{0, 0});
}

// Generic path: any K, any alignment; one workgroup per row, two passes.  Full groups of eight elements move as 16- / 32-byte
// copies without an alignment promise (the compiler picks the access width the target allows), the K % 8 tail and the
// padding columns element by element.
template <int DTYPE, bool TRITON>
__global__ __launch_bounds__(256) void quantize_rows_generic_kernel(
    const void* __restrict__ x, int64_t rows, int64_t K, int64_t in_stride, uint8_t* __restrict__ out,
    int64_t out_stride, float* __restrict__ scale, const float* __restrict__ scale_ub, JaggedRows jag) {
  using elem_t = typename Traits<DTYPE>::elem_t;
  __shared__ uint32_t smem[4];
  const int64_t row = blockIdx.x;
  const elem_t* xr = reinterpret_cast<const elem_t*>(x) + row * in_stride;
  if (!row_is_live(jag, row)) K = 0;   // nothing of the row is read; all codes become zero
  const int64_t nvec = K >> 3;
  const char* xb = reinterpret_cast<const char*>(xr);
  uint32_t m = 0;
  for (int64_t idx = threadIdx.x; idx < nvec; idx += 256) {
    Vec8<DTYPE> v;
    __builtin_memcpy(&v, xb + idx * sizeof(Vec8<DTYPE>), sizeof(Vec8<DTYPE>));
    m = absmax_bits<DTYPE>(m, v);
  }
  m = finish_absmax_bits<DTYPE>(m);
  for (int64_t k = nvec * 8 + threadIdx.x; k < K; k += 256) {
    if constexpr (DTYPE == 2) m = max(m, __float_as_uint(xr[k]) & 0x7FFFFFFFu);
    else m = max(m, (uint32_t)xr[k] & 0x7FFFu);
  }
  m = team_max<256>(m, smem);
  float inv, sc;
  scales_from_amax<DTYPE, TRITON>(Traits<DTYPE>::abs_bits_to_f32(m), scale_ub, jag.triton_eps, inv, sc);
  if (threadIdx.x == 0) scale[row] = sc;
  uint8_t* out_row = out + row * out_stride;
  for (int64_t idx = threadIdx.x; idx < nvec; idx += 256) {
    Vec8<DTYPE> v;
    __builtin_memcpy(&v, xb + idx * sizeof(Vec8<DTYPE>), sizeof(Vec8<DTYPE>));
    const v2u q = quantize_vec8<DTYPE, TRITON, kModeGeneral>(v, inv, 0.f);
    __builtin_memcpy(out_row + idx * 8, &q, 8);
  }
  for (int64_t k = nvec * 8 + threadIdx.x; k < out_stride; k += 256) {
    uint8_t code = 0;
    if (k < K) {
      float f;
      if constexpr (DTYPE == 2) f = xr[k];
      else f = Traits<DTYPE>::to_f32(xr[k]);
      if constexpr (TRITON) f = __builtin_fminf(__builtin_fmaxf(f / inv, -448.0f), 448.0f);
      else f = f * inv;
      code = (uint8_t)(cvt_pk_e4m3fn(f, 0.0f) & 0xFFu);
    }
    out_row[k] = code;
  }
}

// Row-wise dequantization (reference: _kernel_dequantize_fp8_row, fp8_quantize.py:1060-1113):
// out = bf16_rne(fl32(fp8 -> f32) * scale[row]).  1 byte in, 2 bytes out per element: HBM-bound.
//
// A lane converts 8 consecutive codes of one row (K % 8 == 0), so that the 64 stores of a wavefront are 1 KiB without a gap
// (16 codes per lane as two stores left every store instruction with half of each 32 bytes: 8192 x 8192 42.3 -> 32.8 us
// = 6.1 TB/s, 131072 x 128 10.5 -> 9.6; two or four chunks per lane 33.7 and 34.2).  The row is the chunk's index divided by
// the chunks of a row, by a multiply and a shift prepared on the host.  WIDE, from 2^31 chunks on (16 GiB of codes): divides in
// 64 bits and walks the tensor with a grid of bounded size, since one lane per chunk would reach the 2^32 work-items that
// HIP refuses.
struct RowDivider { uint32_t magic, shift; };   // n / d = umulhi(n, magic) >> shift for n < 2^31, d > 1; magic 0: d = 1
template <bool WIDE>
__global__ __launch_bounds__(256) void dequantize_rows_vec_kernel(const uint8_t* __restrict__ xq,
                                                                  const float* __restrict__ scale, int64_t chunks,
                                                                  int64_t chunks_per_row, RowDivider div, uint16_t* __restrict__ out) {
  for (int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x; c < chunks; c += (int64_t)gridDim.x * 256) {
    const v2u q = __builtin_nontemporal_load(reinterpret_cast<const v2u*>(xq) + c);
    int64_t row;
    if constexpr (WIDE) row = c / chunks_per_row;
    else row = div.magic == 0 ? (uint32_t)c : __umulhi((uint32_t)c, div.magic) >> div.shift;
    const float sc = scale[row];
    v4u o;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const auto lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)q[j], false);
      const auto hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)q[j], true);
      o[2 * j] = pack_bf16x2(lo[0] * sc, lo[1] * sc);
      o[2 * j + 1] = pack_bf16x2(hi[0] * sc, hi[1] * sc);
    }
    __builtin_nontemporal_store(o, reinterpret_cast<v4u*>(out) + c);
    if constexpr (!WIDE) break;   // one chunk per lane
  }
}

// Any K, any alignment: a lane takes 8 consecutive codes of the flat tensor; when they lie in one row they move as an
// 8-byte and a 16-byte copy without an alignment promise, otherwise (row boundary, end of the tensor) one by one.
__global__ __launch_bounds__(256) void dequantize_rows_generic_kernel(const uint8_t* __restrict__ xq,
                                                                      const float* __restrict__ scale, int64_t total,
                                                                      int64_t K, uint16_t* __restrict__ out) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  const int64_t chunks = (total + 7) / 8;
  for (int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x; c < chunks; c += stride) {
    const int64_t i0 = c * 8;
    const int n = total - i0 < 8 ? (int)(total - i0) : 8;
    const int64_t r0 = i0 / K;
    if (n == 8 && (i0 + 7) / K == r0) {
      uint32_t w[2];
      __builtin_memcpy(w, xq + i0, 8);
      const float sc = scale[r0];
      uint32_t o[4];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const auto lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)w[i], false);
        const auto hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)w[i], true);
        o[2 * i] = pack_bf16x2(lo[0] * sc, lo[1] * sc);
        o[2 * i + 1] = pack_bf16x2(hi[0] * sc, hi[1] * sc);
      }
      __builtin_memcpy(out + i0, o, 16);
    } else {
      for (int e = 0; e < n; ++e)
        out[i0 + e] = (uint16_t)f32_to_bf16_bits(__builtin_amdgcn_cvt_f32_fp8((int)xq[i0 + e], 0) * scale[(i0 + e) / K]);
    }
  }
}

__global__ void cast_e4m3fn_kernel(const float* __restrict__ in, int64_t n, uint8_t* __restrict__ out) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    out[i] = (uint8_t)(cvt_pk_e4m3fn(in[i], 0.0f) & 0xFFu);
}

template <int DTYPE, bool TRITON>
hipError_t launch_quantize_t(const void* x, int64_t rows, int64_t K, int64_t in_stride, uint8_t* out,
                             int64_t out_stride, float* scale, const float* scale_ub, JaggedRows jag,
                             hipStream_t s) {
  constexpr int ELEM_BYTES = (DTYPE == 2) ? 4 : 2;
  const bool vec_ok = (K % 8 == 0) && (K < (int64_t(1) << 31)) && ((in_stride * ELEM_BYTES) % 16 == 0) &&
                      (reinterpret_cast<uintptr_t>(x) % 16 == 0) && (out_stride % 8 == 0) &&
                      (reinterpret_cast<uintptr_t>(out) % 8 == 0);
  if (!vec_ok) {
    quantize_rows_generic_kernel<DTYPE, TRITON><<<dim3((unsigned)rows), dim3(256), 0, s>>>(
        x, rows, K, in_stride, out, out_stride, scale, scale_ub, jag);
    return hipGetLastError();
  }
  const int k = (int)K;
  const int64_t nvec = K / 8;
  auto team = [&](auto t, auto n) {
    constexpr int TEAM = decltype(t)::value, NV = decltype(n)::value, TEAMS = TEAM > 256 ? 1 : 256 / TEAM;
    const dim3 grid = TEAM <= kWave ? dim3((unsigned)((rows + TEAMS - 1) / TEAMS)) : row_grid(rows);
    if (TEAM >= kWave && nvec <= NV * TEAM - kWave)
      quantize_rows_vec_kernel<DTYPE, TEAM, NV, TRITON, TEAM >= kWave><<<grid, TEAM > 256 ? TEAM : 256, 0, s>>>(
          x, rows, k, in_stride, out, out_stride, scale, scale_ub, jag);
    else
      quantize_rows_vec_kernel<DTYPE, TEAM, NV, TRITON, false><<<grid, TEAM > 256 ? TEAM : 256, 0, s>>>(
          x, rows, k, in_stride, out, out_stride, scale, scale_ub, jag);
    return hipGetLastError();
  };
  // From 2048 rows on the chip is full with a wavefront or less per row: as many lanes as give each one to four vectors,
  // the per-row work (reduction, divisions) then being shared by more elements.  131072 x 128 bf16, Triton arithmetic, by
  // lanes per row: 4 15.3, 8 10.8, 16 11.4, 32 16.2 us; 32768 x 1024: 64 x 2 vectors 16.8, 256 29.9; 8192 x 2048: 64 x 4
  // 9.9, 256 10.8.  Longer rows take a workgroup: 8192 x 4096: 256 x 2 16.7, 64 x 8 17.7, 512 19.4; 8192 x 8192: 256 x 4
  // 30.5, 512 x 2 30.6, 1024 39.9; 4096 x 16384: 512 x 4 31.1, 256 x 8 31.5, 1024 x 2 33.0.
  // Between two steps a workgroup has too many lanes without a vector: 2048 < K <= 2560 takes a wavefront of five (8192 x 2560
  // 9.8, as 256 x 2 11.6; 131072 x 2056 125 / 153, but 131072 x 2560 in torch arithmetic 167 / 157), and 64 < K <= 128 in fp32,
  // whose vectors are twice as wide, 16 lanes of one (1048576 x 72: 77, as 8 x 2 93).
  // (The bounds on the strides keep the byte offsets of a wavefront's up to eight rows between 0 and 2^31; a C caller may walk
  // the input backwards.)
  if (rows >= 2048 && nvec <= 256 && in_stride >= 0 && in_stride * ELEM_BYTES < (1 << 26) && out_stride < (1 << 26)) {
    if (nvec <= 8) return team(Int<8>{}, Int<1>{});
    if (nvec <= 16) return DTYPE == 2 ? team(Int<16>{}, Int<1>{}) : team(Int<8>{}, Int<2>{});
    if (nvec <= 32) return team(Int<16>{}, Int<2>{});
    if (nvec <= 64) return team(Int<32>{}, Int<2>{});
    if (nvec <= 128) return team(Int<64>{}, Int<2>{});
    return team(Int<64>{}, Int<4>{});
  }
  if (rows >= 2048 && nvec > 256 && nvec <= 320) return team(Int<64>{}, Int<5>{});
  if (nvec <= 256) return team(Int<256>{}, Int<1>{});
  if (nvec <= 512) return team(Int<256>{}, Int<2>{});
  if (nvec <= 1024) return team(Int<256>{}, Int<4>{});
  if (nvec <= 2048) return team(Int<512>{}, Int<4>{});
  if (nvec <= 4096) return team(Int<1024>{}, Int<4>{});
  if (DTYPE != 2 && nvec <= 8192) return team(Int<1024>{}, Int<(DTYPE != 2 ? 8 : 1)>{});
  quantize_rows_long_kernel<DTYPE, TRITON><<<(unsigned)rows, 256, 0, s>>>(x, rows, k, in_stride, out, out_stride, scale, scale_ub, jag);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_quantize_fp8_row(const void* x, int dtype, int64_t rows, int64_t K, int64_t in_stride,
                                   void* xq, int64_t K_out, float* scale, const float* scale_ub,
                                   const void* zero_start, int zero_start_is_i32, int64_t rows_per_group,
                                   int triton_arithmetic, float triton_eps, hipStream_t s) {
  uint8_t* out = reinterpret_cast<uint8_t*>(xq);
  const JaggedRows jag{zero_start, rows_per_group > 0 ? rows_per_group : 1, zero_start_is_i32, triton_eps};
  if (triton_arithmetic) {
    switch (dtype) {
      case 0: return launch_quantize_t<0, true>(x, rows, K, in_stride, out, K_out, scale, scale_ub, jag, s);
      case 1: return launch_quantize_t<1, true>(x, rows, K, in_stride, out, K_out, scale, scale_ub, jag, s);
      default: return launch_quantize_t<2, true>(x, rows, K, in_stride, out, K_out, scale, scale_ub, jag, s);
    }
  }
  switch (dtype) {
    case 0: return launch_quantize_t<0, false>(x, rows, K, in_stride, out, K_out, scale, scale_ub, jag, s);
    case 1: return launch_quantize_t<1, false>(x, rows, K, in_stride, out, K_out, scale, scale_ub, jag, s);
    default: return launch_quantize_t<2, false>(x, rows, K, in_stride, out, K_out, scale, scale_ub, jag, s);
  }
}

hipError_t launch_dequantize_fp8_row(const void* xq, const float* scale, int64_t rows, int64_t K, void* out,
                                     hipStream_t s) {
  const int64_t total = rows * K;
  if (total <= 0) return hipSuccess;
  if (K % 8 == 0 && reinterpret_cast<uintptr_t>(xq) % 8 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0) {
    const uint8_t* in = reinterpret_cast<const uint8_t*>(xq);
    uint16_t* dst = reinterpret_cast<uint16_t*>(out);
    const int64_t chunks = total / 8, per_row = K / 8, blocks = (chunks + 255) / 256;
    RowDivider div{0, 0};
    if (chunks >= (int64_t(1) << 31)) {
      dequantize_rows_vec_kernel<true><<<1u << 16, 256, 0, s>>>(in, scale, chunks, per_row, div, dst);
    } else {
      if (per_row > 1) {   // 2^shift < d <= 2^(shift + 1): magic = ceil(2^(32 + shift) / d) < 2^32, exact for n < 2^31
        while ((int64_t(2) << div.shift) < per_row) ++div.shift;
        div.magic = (uint32_t)(((uint64_t(1) << (32 + div.shift)) + per_row - 1) / per_row);
      }
      dequantize_rows_vec_kernel<false><<<(unsigned)blocks, 256, 0, s>>>(in, scale, chunks, per_row, div, dst);
    }
  } else {
    const int64_t want = ((total + 7) / 8 + 255) / 256;
    const unsigned blocks = (unsigned)(want > 65536 ? 65536 : want);
    dequantize_rows_generic_kernel<<<blocks, 256, 0, s>>>(reinterpret_cast<const uint8_t*>(xq), scale, total, K,
                                                         reinterpret_cast<uint16_t*>(out));
  }
  return hipGetLastError();
}

hipError_t launch_cast_e4m3fn(const float* in, int64_t n, void* out, hipStream_t s) {
  const int64_t want = (n + 255) / 256;
  const unsigned blocks = (unsigned)(want < 1 ? 1 : (want > 65536 ? 65536 : want));
  cast_e4m3fn_kernel<<<blocks, 256, 0, s>>>(in, n, reinterpret_cast<uint8_t*>(out));
  return hipGetLastError();
}

}  // namespace mslk_amd
