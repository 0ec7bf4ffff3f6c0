// Row access of the row-wise kernels (quantizer, fused producers): buffer loads and stores, and the team maximum.
//
// Why buffer instructions.  A lane owns a fixed number of 16-byte vectors of its row, of which the last may lie beyond the
// row's end.  Guarded by a branch per vector, each load ends up in a block of its own whose end waits for it: a row of eight
// vectors then costs eight round trips to memory one after the other (4096 x 4096 bf16: 12.1 us).  A buffer load checks
// the offset against the descriptor's size itself and returns zero beyond it without touching memory, so the loads of a
// row are one straight run of instructions, all in flight at once; stores beyond the end are dropped the same way.
#pragma once
#include "common.h"

namespace mslk_amd {

typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef __amdgpu_buffer_rsrc_t buffer_t;

template <int N> struct Int { static constexpr int value = N; };   // a template argument carried by a value

constexpr uint32_t kBeyondBuffer = 0x80000000u;   // an offset no descriptor made here reaches (sizes stay below 2^31)
constexpr int kCacheNt = 2, kCacheSc1 = 16;       // cache policy bits of the buffer instructions: non-temporal, system scope

// HIP refuses a launch of 2^32 or more work-items along one dimension: of workgroups of 1024 lanes that hold a row each, 2^22
// rows.  From 2^21 workgroups on the grid goes on along y, the last line of it beyond the rows.
constexpr int64_t kRowGridX = int64_t(1) << 21;
inline dim3 row_grid(int64_t blocks) {
  return blocks <= kRowGridX ? dim3((unsigned)blocks) : dim3((unsigned)kRowGridX, (unsigned)((blocks + kRowGridX - 1) / kRowGridX));
}
MSLK_AMD_DEVINL int64_t row_block() { return blockIdx.y * (uint32_t)kRowGridX + blockIdx.x; }

// `base` and `bytes` have to be the same in every lane of the wavefront.
MSLK_AMD_DEVINL buffer_t make_buffer(const void* base, uint32_t bytes) {
  const uint64_t v = reinterpret_cast<uint64_t>(base);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)v), hi = __builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(((uint64_t)hi << 32) | lo), 0,
                                           __builtin_amdgcn_readfirstlane((int)bytes), 0x00020000);
}
// Read-once input: non-temporal.
MSLK_AMD_DEVINL v4u buffer_load16(buffer_t b, uint32_t off) {
  return __builtin_amdgcn_raw_buffer_load_b128(b, (int)off, 0, kCacheNt);
}
// Codes: written through at system scope, as store8_write_through() (common.h) does and for its reasons.
MSLK_AMD_DEVINL void buffer_store8_through(buffer_t b, uint32_t off, v2u v) {
  __builtin_amdgcn_raw_buffer_store_b64(v, b, (int)off, 0, kCacheSc1);
}

template <int CTRL>
MSLK_AMD_DEVINL uint32_t dpp_max(uint32_t m) {
  return max(m, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, CTRL, 0xF, 0xF, true));
}
// Maximum over aligned groups of TEAM lanes, in every lane of the group; TEAM > 64: over the workgroup of TEAM lanes, one
// word of `smem` per wavefront.  Inside 16 lanes by data-parallel moves (a handful of cycles each, where a shuffle through
// LDS takes about a hundred), across 64 through scalar registers.
template <int TEAM>
MSLK_AMD_DEVINL uint32_t team_max(uint32_t m, uint32_t* smem) {
  if constexpr (TEAM >= 2) m = dpp_max<0xB1>(m);     // lanes 1 0 3 2 of a quad
  if constexpr (TEAM >= 4) m = dpp_max<0x4E>(m);     // lanes 2 3 0 1
  if constexpr (TEAM >= 8) m = dpp_max<0x141>(m);    // mirrored inside 8 lanes
  if constexpr (TEAM >= 16) m = dpp_max<0x140>(m);   // mirrored inside 16 lanes
  if constexpr (TEAM == 32) m = max(m, (uint32_t)__shfl_xor((int)m, 16, 64));
  if constexpr (TEAM >= 64) {
    const uint32_t a = max((uint32_t)__builtin_amdgcn_readlane((int)m, 0), (uint32_t)__builtin_amdgcn_readlane((int)m, 16));
    const uint32_t b = max((uint32_t)__builtin_amdgcn_readlane((int)m, 32), (uint32_t)__builtin_amdgcn_readlane((int)m, 48));
    m = max(a, b);
  }
  if constexpr (TEAM > 64) {
    if ((threadIdx.x & 63) == 0) smem[threadIdx.x >> 6] = m;
    __syncthreads();
    uint32_t w = smem[0];
#pragma unroll
    for (int i = 1; i < TEAM / 64; ++i) w = max(w, smem[i]);
    m = (uint32_t)__builtin_amdgcn_readfirstlane((int)w);
  }
  return m;
}

}  // namespace mslk_amd
