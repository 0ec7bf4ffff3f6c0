// Kernels of the grouped GEMM whose group extents live in device memory (or are uniform), with the tile order they share
// with the TensorList kernel.  Included by the translation units that instantiate the layouts (gemm_grouped.hip: row blocks
// given by sizes or offsets, and the TensorList form; gemm_grouped_layouts.hip: offsets over N and K, padded rows;
// gemm_grouped_uniform.hip: the uniform batch with its bias variants), so that they compile side by side.
#pragma once
#include "gemm_tile.h"
#include "kernels.h"
#include "rows.h"

namespace mslk_amd {
namespace {


constexpr int kXcds = 8;
constexpr int kGroupM = 4;

// Tile order inside one group: panels of kGroupM row tiles, column-major inside a panel.  Returns the number of row tiles
// of the tile's panel: the tiles that read one weight block at about the same time.
MSLK_AMD_DEVINL int local_tile(int t, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int panel = kGroupM * tiles_n;
  const int first_m = (t / panel) * kGroupM;
  const int rows = tiles_m - first_m < kGroupM ? tiles_m - first_m : kGroupM;
  tm = first_m + (t % panel) % rows;
  tn = (t % panel) / rows;
  return rows;
}

// Groups whose extents live in device memory (or are uniform).  `layout` says which dimension varies
// per group and how it is encoded; the fixed dimensions come from p.M / p.N / p.K, where the varying
// one holds the total over all groups.
//   kGroupsSizesM    int64 sizes of the row blocks of XQ [sum M, K]; WQ [G, N, K]; Y [sum M, N]
//   kGroupsOffsetsM  int32 cumulative ends of the same row blocks
//   kGroupsOffsetsN  XQ [G, M, K]; int32 cumulative ends of row blocks of WQ [sum N, K]; Y [M, sum N]
//   kGroupsOffsetsK  XQ [M, sum K], WQ [N, sum K]; int32 cumulative ends of K slices; Y [G, M, N]
//   kGroupsUniform   XQ [G, M, K], WQ [G, N, K], Y [G, M, N]
//   kGroupsPrepadM   as uniform, but only the first layout[g] (int64) rows of group g are computed
// Scales follow the operand they belong to ([sum M] or [G, M]; [sum N] or [G, N]).
struct GroupSpan {
  int gi;        // group
  int64_t o0;    // first index of the group along the varying dimension
  int len;       // extent of the group along the varying dimension
  int t;         // tile index inside the group
};

MSLK_AMD_DEVINL int64_t uniform64(int64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)v), hi = __builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// x + y for 0 <= x, y < 2^31, at most 2^31 - 1 (one unsigned addition cannot wrap): sizes that add up to more than a tensor
// holds always end beyond it.
MSLK_AMD_DEVINL int saturating_sum(int x, int y) {
  const uint32_t u = (uint32_t)x + (uint32_t)y;
  return (int)(u > 0x7FFFFFFFu ? 0x7FFFFFFFu : u);
}
// Inclusive prefix sum over the 64 lanes of non-negative values by data-parallel moves: inside each row of 16 lanes, then
// the last lane of rows 0 and 2 added to rows 1 and 3, then lane 31 to rows 2 and 3.  Lanes without a source add zero.
template <bool SATURATE, int CTRL, int ROWS>
MSLK_AMD_DEVINL int prefix_step(int v) {
  const int o = __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xF, false);
  return SATURATE ? saturating_sum(v, o) : v + o;
}
template <bool SATURATE>
MSLK_AMD_DEVINL int wave_prefix_sum(int v) {
  v = prefix_step<SATURATE, 0x111, 0xF>(v);   // one lane to the right
  v = prefix_step<SATURATE, 0x112, 0xF>(v);   // two
  v = prefix_step<SATURATE, 0x114, 0xF>(v);   // four
  v = prefix_step<SATURATE, 0x118, 0xF>(v);   // eight
  v = prefix_step<SATURATE, 0x142, 0xA>(v);   // lane 15 of a row to the next row
  return prefix_step<SATURATE, 0x143, 0xC>(v);   // lane 31 to the upper half
}

// Workgroup -> (group, tile of the group) where the groups are K slices: every group has the same `per` output tiles, but a
// tile costs what its slice is long.  Two orders:
// - in group order, every XCD an equal run of tiles: whole groups, whose operands only that XCD's L2 fetches;
// - groups by falling length (the longest tiles start first, the short ones fill the end), dealt to the XCDs in runs of
//   per / 8 tiles, so that every XCD gets the same share of every group and a run still holds neighbouring tiles.  Groups
//   beyond the first 64 keep their order behind the sorted ones.
// The second where the first gives one XCD much more than the others: eight [4096 x 2048] gradients over 16384 rows, group
// sizes falling like 1 / rank^1.1, 363 -> 156 us, because one XCD owned the whole longest group.  The first otherwise: with
// equal groups the second, whose operands every XCD fetches, is slower (16 x [1024 x 1024] over 16384 rows: 19.5 / 23.6 us,
// 16 x [1408 x 2880] 81 / 91, 32 x [4096 x 2048] over 8192 152 / 177), and so it is with few tiles per group (32 x [1024 x
// 1024] over 32768 rows of sizes like 1 / rank^1.1: 89 / 104).
// Every workgroup decides alike from the lengths (k_slices_in_order).
MSLK_AMD_DEVINL int k_slice_run(int per) { return per > kXcds ? (per + kXcds - 1) / kXcds : 1; }

// Whether the first order serves.  A tile costs its slice's length plus kTileCost, which is about what its output takes.  Of G / 8
// groups an XCD gets in the first order the longest one sets the pace; the order serves while that XCD has at most a fifth
// more than its share (beyond 64 groups, where the second sorts only some of them, a half).  It also serves where the second
// order leaves a run of fewer than four neighbouring tiles, or none wait for a CU.
MSLK_AMD_DEVINL bool k_slices_in_order(const DeviceGroups& p, int per, int per_xcd, int lane_begin, int lane_end) {
  constexpr float kTileCost = 512.f;
  if (p.G == 1 || per < 32 || per_xcd <= 32) return true;
  const int32_t* off = static_cast<const int32_t*>(p.layout);
  const int lane = threadIdx.x & 63;
  auto length = [](int begin, int end) {   // of a consistent slice; anything else counts as none
    const int len = (int)((uint32_t)end - (uint32_t)begin);
    return len < 0 ? 0 : len;
  };
  int longest = length(lane_begin, lane_end);
  for (int gi = 64 + lane; gi < p.G; gi += 64) {
    const int len = length(off[gi - 1], off[gi]);
    longest = len > longest ? len : longest;
  }
  const float most = (float)team_max<64>((uint32_t)longest, nullptr) + kTileCost, groups = (float)p.G;
  const float all = (float)p.K + groups * kTileCost;
  return (most * groups - all) * 8.f <= (p.G <= 64 ? 0.2f : 0.5f) * (groups < 8.f ? 8.f : groups) * all;
}

MSLK_AMD_DEVINL bool k_slice_tile(const DeviceGroups& p, int wg, int per, int& group, int& tile, int64_t& begin, int64_t& end) {
  const int32_t* off = static_cast<const int32_t*>(p.layout);
  const int lane = threadIdx.x & 63, total = p.G * per, per_xcd = (total + kXcds - 1) / kXcds;
  const int lane_begin = lane && lane < p.G ? off[lane - 1] : 0, lane_end = lane < p.G ? off[lane] : 0;
  int gi;
  if (k_slices_in_order(p, per, per_xcd, lane_begin, lane_end)) {
    const int at = wg % kXcds * per_xcd + wg / kXcds;
    if (wg / kXcds >= per_xcd || at >= total) return false;
    gi = at / per;
    tile = __builtin_amdgcn_readfirstlane(at - gi * per);
  } else {
    const int run = k_slice_run(per), slot = wg / kXcds;
    const int at = (slot / run * kXcds + wg % kXcds) * run + slot % run;
    gi = at / per;
    if (gi >= p.G) return false;
    tile = __builtin_amdgcn_readfirstlane(at - gi * per);
    if (gi < 64) {   // the group of rank gi: lane i holds the length of group i, its rank is the number of groups in front of it
      const int n = p.G < 64 ? p.G : 64;
      const int raw = (int)((uint32_t)lane_end - (uint32_t)lane_begin);
      const int len = lane < n ? (raw < 0 ? -1 : raw) : INT32_MIN;   // lanes without a group are in front of none
      int ahead = 0;
      for (int j = 0; j < n; j += 8) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const int other = __builtin_amdgcn_readlane(len, j + k);
          ahead += (other > len || (other == len && j + k < lane)) ? 1 : 0;
        }
      }
      gi = __ffsll((long long)__ballot(lane < n && ahead == gi)) - 1;
    }
  }
  gi = __builtin_amdgcn_readfirstlane(gi);
  group = gi;
  if (gi < 64) {
    begin = __builtin_amdgcn_readlane(lane_begin, gi);
    end = __builtin_amdgcn_readlane(lane_end, gi);
  } else {
    begin = off[gi - 1];
    end = off[gi];
  }
  return true;
}

// Groups of rows (or of columns) by sizes or offsets: the tile list of a launch, and the group a tile of it belongs to.
// The G extents are read 64 at a time, one per lane, and turned into tile ranges by a wave-level prefix sum, so the
// lookup costs one memory round trip for up to 128 groups (the first two chunks are fetched together and stay in
// registers) instead of G dependent ones.  A workgroup of 256 x 256 tiles holds its CU's whole LDS, so nothing else runs
// under its lookup (two of 128 x 128 share a CU): with more round trips for the groups beyond 64 and sums through LDS shuffles (a hundred cycles per step) 128 experts x
// 2048 x 768 took 65.5 us over 8192 rows and 120.0 over 32768 (now 56.3 and 114.8), 64 x 4096 x 1024 over 16384 128.4
// (120.1), 16 x 8192 x 5120 over 8192 324 (323).
// The total tile count is formed first: XCD x (workgroup id mod 8) then takes a contiguous slice of the tile list, so
// that the row tiles of a group that share a weight panel run on one XCD and find it in its L2 (without the slices the
// device-extent layouts fetched 1.6 times what the host-extent kernel fetches for the same 16 experts).
template <int LAYOUT, int BM, int BN>
struct BlockGroups {
  // Every quantity fits 32 bits (the host checks the dimensions and the grid): sizes beyond the tensor mark the group bad.
  struct Extent { int64_t size; int begin, end; };
  struct Chunk { int start, len, tiles, incl; };
  Chunk c0, c1;
  int carry_len2;        // of the first 128 groups, for the chunks beyond them
  bool seen_bad2;
  int64_t total_tiles;   // of the launch
  int64_t per_xcd;       // of an XCD's slice

  MSLK_AMD_DEVINL static Extent fetch(const DeviceGroups& p, int base) {
    Extent x{0, 0, 0};
    const int gi = base + (threadIdx.x & 63);
    if (gi < p.G) {
      if constexpr (LAYOUT == kGroupsSizesM) {
        x.size = static_cast<const int64_t*>(p.layout)[gi];
      } else {
        x.begin = gi ? static_cast<const int32_t*>(p.layout)[gi - 1] : 0;
        x.end = static_cast<const int32_t*>(p.layout)[gi];
      }
    }
    return x;
  }
  // `seen_bad` carries "an earlier group was inconsistent" from chunk to chunk: such a group and every group after it
  // own no tiles, so the tile count, the XCD slices and the lookup all stop at the first bad group and every tile
  // of the groups in front of it gets a workgroup (the grid is sized for consistent extents).
  MSLK_AMD_DEVINL static Chunk chunk_of(const DeviceGroups& p, const Extent& x, int base, int& carry_len, bool& seen_bad) {
    const int fixed_tiles = LAYOUT == kGroupsOffsetsN ? (p.M + BM - 1) / BM : (p.N + BN - 1) / BN;
    const int blk = LAYOUT == kGroupsOffsetsN ? BN : BM;
    const int64_t total = LAYOUT == kGroupsOffsetsN ? p.N : p.M;
    const int lane = threadIdx.x & 63;
    Chunk c;
    const bool in = base + lane < p.G;
    bool bad;
    if constexpr (LAYOUT == kGroupsSizesM) {
      bad = x.size < 0 || x.size > total;
      c.len = bad ? 0 : (int)x.size;
      const int end = saturating_sum(carry_len, wave_prefix_sum<true>(c.len));
      c.start = end - c.len;
      carry_len = __builtin_amdgcn_readlane(end, 63);
      bad = bad || (in && (end > total || end == 0x7FFFFFFF));
    } else {
      const int64_t len64 = (int64_t)x.end - x.begin;
      bad = len64 < 0 || x.begin < 0 || x.end > total;
      c.start = x.begin;
      c.len = bad ? 0 : (int)len64;
    }
    const unsigned long long bad_lanes = __ballot(bad);
    const bool after_bad = seen_bad || (bad_lanes != 0 && lane >= __ffsll((long long)bad_lanes) - 1);
    seen_bad = seen_bad || bad_lanes != 0;
    c.tiles = (in && !after_bad) ? ((c.len + blk - 1) / blk) * fixed_tiles : 0;
    c.incl = wave_prefix_sum<false>(c.tiles);
    return c;
  }
  MSLK_AMD_DEVINL static int tiles_of(const Chunk& c) { return __builtin_amdgcn_readlane(c.incl, 63); }

  MSLK_AMD_DEVINL void scan(const DeviceGroups& p) {
    const Extent x0 = fetch(p, 0), x1 = fetch(p, 64);
    int carry_len = 0;
    bool seen_bad = false;
    c0 = chunk_of(p, x0, 0, carry_len, seen_bad);
    c1 = chunk_of(p, x1, 64, carry_len, seen_bad);   // no groups there: no tiles
    carry_len2 = carry_len;
    seen_bad2 = seen_bad;
    total_tiles = (int64_t)tiles_of(c0) + tiles_of(c1);
    for (int base = 128; base < p.G && !seen_bad; base += 64)
      total_tiles += tiles_of(chunk_of(p, fetch(p, base), base, carry_len, seen_bad));
    per_xcd = (total_tiles + kXcds - 1) / kXcds;
  }
  // Group, extent and place inside the group of tile `tile` < total_tiles of the list.
  MSLK_AMD_DEVINL bool find(const DeviceGroups& p, int64_t tile, GroupSpan& sp) const {
    int64_t carry_tiles = 0;
    auto find_in = [&](const Chunk& c, int base) {
      const int64_t excl = carry_tiles + c.incl - c.tiles;
      const unsigned long long hit = __ballot(c.tiles > 0 && tile >= excl && tile < excl + c.tiles);
      if (hit == 0) {
        carry_tiles += tiles_of(c);
        return false;
      }
      const int src = __ffsll((long long)hit) - 1;
      // the results are the same in every lane: out of scalar registers, so that the tile's addresses live there
      sp.gi = base + src;
      sp.o0 = __builtin_amdgcn_readlane(c.start, src);
      sp.len = __builtin_amdgcn_readlane(c.len, src);
      sp.t = (int)(uniform64(tile - carry_tiles) - __builtin_amdgcn_readlane(c.incl - c.tiles, src));
      return true;
    };
    if (find_in(c0, 0) || find_in(c1, 64)) return true;
    int carry_len = carry_len2;
    bool seen_bad = seen_bad2;
    for (int base = 128; base < p.G && !seen_bad; base += 64)
      if (find_in(chunk_of(p, fetch(p, base), base, carry_len, seen_bad), base)) return true;
    return false;
  }
  // The same for a tile per lane (all lanes of the wavefront call it; `live`: the lane has a tile).
  MSLK_AMD_DEVINL void find_lanes(const DeviceGroups& p, int tile, bool live, int& gi, int& start, int& len, int& t) const {
    int carry_tiles = 0;
    auto find_in = [&](const Chunk& c, int base) {
      const int rel = tile - carry_tiles, n = tiles_of(c);
      int pos = 0;   // groups of the chunk whose tiles end at or before `rel`
#pragma unroll
      for (int step = 32; step > 0; step >>= 1) pos += __shfl(c.incl, pos + step - 1, 64) <= rel ? step : 0;
      const int s = __shfl(c.start, pos, 64), l = __shfl(c.len, pos, 64), before = __shfl(c.incl - c.tiles, pos, 64);
      if (rel >= 0 && rel < n) { gi = base + pos; start = s; len = l; t = rel - before; }
      carry_tiles += n;
    };
    gi = start = len = t = 0;
    find_in(c0, 0);
    if (p.G > 64) find_in(c1, 64);
    int carry_len = carry_len2;
    bool seen_bad = seen_bad2;
    for (int base = 128; base < p.G && !seen_bad && __ballot(live && tile >= carry_tiles) != 0; base += 64)
      find_in(chunk_of(p, fetch(p, base), base, carry_len, seen_bad), base);
  }
};

template <int LAYOUT, int BM, int BN>
MSLK_AMD_DEVINL bool find_group(const DeviceGroups& p, int t, GroupSpan& sp) {
  const int tiles_m = (p.M + BM - 1) / BM, tiles_n = (p.N + BN - 1) / BN;
  if constexpr (LAYOUT == kGroupsOffsetsK) {
    const int per = tiles_m * tiles_n;
    int64_t b, e;
    if (!k_slice_tile(p, t, per, sp.gi, sp.t, b, e)) return false;
    sp.o0 = b;
    sp.len = (int)(e - b);
    return b >= 0 && e >= b && e <= p.K;
  } else if constexpr (LAYOUT == kGroupsUniform || LAYOUT == kGroupsPrepadM) {
    const int per = tiles_m * tiles_n;
    sp.gi = t / per;
    sp.t = t - sp.gi * per;
    if (sp.gi >= p.G) return false;
    if constexpr (LAYOUT == kGroupsUniform) {
      sp.o0 = 0;
      sp.len = 0;
      return true;
    } else {
      const int64_t live = static_cast<const int64_t*>(p.layout)[sp.gi];
      sp.o0 = 0;
      sp.len = (int)(live < 0 ? 0 : (live > p.M ? p.M : live));
      return true;
    }
  } else {
    BlockGroups<LAYOUT, BM, BN> groups;
    groups.scan(p);
    const int64_t slot = t / kXcds;                       // `t` arrives as the workgroup id
    const int64_t tile = (int64_t)(t % kXcds) * groups.per_xcd + slot;
    if (slot >= groups.per_xcd || tile >= groups.total_tiles) return false;
    return groups.find(p, tile, sp);
  }
}

// Scalar tile for operands the DMA path cannot fetch (row starts or K extents that are not multiples
// of 16 bytes): one lane per output element, sequential K.
template <int BM, int BN, int BIAS>
MSLK_AMD_DEVINL void slow_tile(const uint8_t* a, const uint8_t* b, const float* xs, const float* ws,
                               const void* bias, uint16_t* y, int m_rem, int n_rem, int ldc, int K, int64_t ld) {
  const int mt = m_rem < BM ? m_rem : BM, nt = n_rem < BN ? n_rem : BN;
  for (int idx = threadIdx.x; idx < mt * nt; idx += 256) {
    const int m = idx / nt, n = idx - m * nt;
    const uint8_t* ar = a + m * ld;
    const uint8_t* br = b + n * ld;
    float acc = 0.f;
    for (int k = 0; k < K; ++k)
      acc += __builtin_amdgcn_cvt_f32_fp8((int)ar[k], 0) * __builtin_amdgcn_cvt_f32_fp8((int)br[k], 0);
    float v = (acc * ws[n]) * xs[m];
    if constexpr (BIAS == 1) v += static_cast<const float*>(bias)[n];
    if constexpr (BIAS == 2) v += bf16_bits_to_f32(static_cast<const uint16_t*>(bias)[n]);
    y[(int64_t)m * ldc + n] = (uint16_t)f32_to_bf16_bits(v);
  }
}

// 256 x 256 tiles of row groups: one workgroup per CU walks its share of the tile list, tile after tile in one chain of K steps
// (GemmTile::chain_tile).
using RowTileShape = TileShape<256, 256>;
struct RowTile {
  const uint8_t *a, *b;
  const float *xs, *ws;
  uint16_t* y;
  int m_rem, n_rem;   // valid rows / columns from the tile's first
  int N, K;           // row pitch of Y, bytes of an operand row
  int stream;         // the only reader of its weight block at that time: weights fetched with non-temporal loads
};

// Division of the `tiles` tiles of an XCD among its `wgs` workgroups.  The first `wgs` workgroups walk the full passes, one entry of
// the slice each per pass.  What is left over for a last pass, as long as it is at most three quarters of one, is
// given to further workgroups, one tile each, which the hardware starts where one of the first ones ends: tiles cost what their
// rows cost, and the workgroups that were given cheap ones take what is left.  At most a quarter of a pass is cut into quarters of tiles besides.
// (16 experts x 5120 x 4096 over 8192 skewed rows, 780 tiles: a fourth pass with 12 of 256 workgroups busy 184 us, left-over tiles whole 185, in
// quarters 167; 64 groups, 16384 rows x 2816 x 2880 204 / 198 / 197.)
// Neighbouring entries are the row tiles of a panel (local_tile), the last of which may be ragged.  From pass to pass a workgroup
// moves on by wgs + turn entries, and wgs + turn has no divisor in common with any number of row tiles in a panel: every workgroup gets
// its share of the ragged ones.  With entry i for workgroup i % wgs half of the 32 workgroups of an XCD were given all full tiles
// of groups of 300 rows, and the launch took as long as full tiles do (64 x 300 rows x 4096 x 2048: 215 us, now 194; 128 x 257 x 2048 x 768
// 112 / 92; 16 x 257 x 8192 x 2048 107 / 97; skewed sizes the same within 2 %).
struct SliceShares {
  int wgs, turn;
  int walked;        // entries of the slice that the first workgroups walk
  int pieces;        // of a left-over tile: 1 or 4
  __host__ __device__ SliceShares(int tiles, int workgroups) : wgs(workgroups) {
    static_assert(kGroupM <= 4, "one to four row tiles in a panel");
    const int left = tiles % wgs;
    const bool apart = tiles > wgs && left * 4 <= wgs * 3;
    walked = apart ? tiles - left : tiles;
    pieces = left * 4 <= wgs ? 4 : 1;
    const int r = wgs % 6;
    turn = r == 2 ? 3 : r == 3 ? 2 : r == 1 || r == 5 ? 0 : 1;   // wgs + turn is 1 or 5 modulo 6
  }
  // Entry of the slice that workgroup `worker` < wgs walks in `pass`: its own if it is below `walked`.
  __host__ __device__ int walked_entry(int worker, int pass) const { return pass * wgs + (worker + pass * turn) % wgs; }
  // Every workgroup with work has one whole tile: the chain gains nothing.
  __host__ __device__ bool no_second_tile(int tiles) const { return tiles <= wgs || (walked <= wgs && pieces == 1); }
  // Left-over entry, and piece of it, of workgroup `worker` >= wgs: one of the slice if it is below `tiles`.
  __host__ __device__ int left_entry(int worker) const { return walked + (worker - wgs) / pieces; }
  __host__ __device__ int left_piece(int worker) const { return (worker - wgs) % pieces; }
};

// The tiles of one workgroup, found 64 at a time, one per lane: row and column, group and what is left of it.
struct TileBatch {
  int row, m_rem, col, group, stream, count;
};

// What the chain takes: 16-byte pieces of the rows of all operands, of the column scales and of Y, and three K steps.  (Of operands that
// are not marked unaligned: its offsets inside a tile have 32 bits.)
inline bool chain_takes(int64_t N, int64_t K, const void* xq, const void* wq, const void* ws, const void* y) {
  const uintptr_t all = reinterpret_cast<uintptr_t>(xq) | reinterpret_cast<uintptr_t>(wq) | reinterpret_cast<uintptr_t>(ws) | reinterpret_cast<uintptr_t>(y);
  return K > 2 * kBK && K % 16 == 0 && N % 8 == 0 && all % 16 == 0;
}

// One of four pieces of a tile, by a workgroup of its own.
MSLK_AMD_DEVINL void run_quarter_tile(char* lds, const RowTile& t, int piece) {
  using TS = TileShape<128, 128, 2, 2, 5>;
  const int row = (piece & 1) * 128, col = (piece >> 1) * 128;
  if (row >= t.m_rem || col >= t.n_rem) return;
  GemmTile<TS, 0> tile;
  tile.run(lds, t.a + (int64_t)row * t.K, t.b + (int64_t)col * t.K, t.xs + row, t.ws + col, nullptr, t.y + (int64_t)row * t.N + col,
           t.m_rem - row, t.n_rem - col, t.N, t.K);
}

// Tile `t` and then those that `next(tile)` gives, one after the other.
template <typename Next>
MSLK_AMD_DEVINL void walk_row_tiles(char* lds, RowTile t, Next&& next) {
  using TS = RowTileShape;
  using Plain = GemmTile<TS, 0, false, true, TS::LA / 2, false, false, true>;
  using Streamed = GemmTile<TS, 0, false, true, TS::LA / 2, false, true, true>;
  RowTile n;
  auto operands = [](const RowTile& w) { return TileOperands{w.a, w.b, w.m_rem, w.n_rem, (uint32_t)w.K}; };
  Plain tile;
  Streamed streamed;
  TileChain<TS> chain(lds);
  tile.chain_start(chain, operands(t));
  bool more = next(n);   // under the first loads
  tile.chain_started();
  for (;;) {
    if (!more) {   // the last two steps issue loads all the same: of one row of each operand, which the caches hold
      n = t;
      n.m_rem = n.n_rem = 1;
    }
    const TileOperands o = operands(n);
    // One K loop and epilogue per number of m fragments with valid rows and kind of weight loads: a common end for all would
    // have the sums moved between registers.
    auto run = [&](auto& build, auto fragments, auto all) {
      constexpr int FMV = decltype(fragments)::value;
      v4f acc[TS::FN][TS::FM];
      TileScales<TS> scales;
      build.template chain_tile<FMV>(chain, t.K, o, acc, scales, t.xs, t.ws, t.m_rem, t.n_rem);
      build.template epilogue_direct<decltype(all)::value != 0, FMV>(acc, scales, t.y, t.m_rem, t.n_rem, t.N);
    };
    auto run_rows = [&](auto& build) {
      constexpr int Q = TS::kBM / 4, FM = TS::FM;
      if (t.m_rem >= TS::kBM && t.n_rem >= TS::kBN) run(build, Int<FM>(), Int<1>());
      else if (t.m_rem > 3 * Q) run(build, Int<FM>(), Int<0>());
      else if (t.m_rem > 2 * Q) run(build, Int<3 * FM / 4>(), Int<0>());
      else if (t.m_rem > Q) run(build, Int<FM / 2>(), Int<0>());
      else run(build, Int<FM / 4>(), Int<0>());
    };
    if (t.stream) {
      streamed.adopt(tile);
      run_rows(streamed);
      tile.adopt(streamed);
    } else {
      run_rows(tile);
    }
    if (!more) break;
    t = n;
    more = next(n);
  }
  wait_vmcnt0();   // no copy into LDS may outlive the workgroup
}

// `wgs`: workgroups per XCD that walk the full passes; up to as many more of them take what is left.
template <int LAYOUT>
__global__ __launch_bounds__(256) void grouped_rows_kernel(DeviceGroups p, int wgs) {
  using TS = RowTileShape;
  constexpr int BM = TS::kBM, BN = TS::kBN;
  __shared__ __attribute__((aligned(1024))) char lds[TS::LDS_BYTES];
  BlockGroups<LAYOUT, BM, BN> groups;
  groups.scan(p);
  const int xcd = blockIdx.x % kXcds, per_xcd = (int)groups.per_xcd, left = (int)groups.total_tiles - xcd * per_xcd;
  const int tiles = left < per_xcd ? left : per_xcd;
  const SliceShares shares(tiles, wgs);
  const int worker = blockIdx.x / kXcds;
  const bool rest = worker >= wgs;
  auto tile_at = [&](int64_t group, int64_t row, int m_rem, int64_t col, int stream, RowTile& w) {
    w.m_rem = m_rem;
    w.stream = stream;
    w.n_rem = p.N - (int)col;
    w.a = p.xq + row * p.K;
    w.b = p.wq + (group * p.N + col) * p.K;
    w.xs = p.xs + row;
    w.ws = p.ws + group * p.N + col;
    w.y = p.y + row * p.N + col;
    w.N = p.N;
    w.K = p.K;
  };
  // The first tile, often the only one, is found for itself; the others, 64 at a time, under its first loads.
  const int entry = rest ? shares.left_entry(worker) : shares.walked_entry(worker, 0);
  GroupSpan sp;
  if (entry >= (rest ? tiles : shares.walked) || !groups.find(p, (int64_t)xcd * per_xcd + entry, sp)) return;
  RowTile t;
  {
    int tm, tn;
    const int stream = local_tile(sp.t, (sp.len + BM - 1) / BM, (p.N + BN - 1) / BN, tm, tn) == 1;
    tile_at(sp.gi, sp.o0 + tm * BM, sp.len - tm * BM, tn * BN, stream, t);
  }
  if (rest && shares.pieces > 1) {
    run_quarter_tile(lds, t, shares.left_piece(worker));
    return;
  }
  TileBatch b;
  int i = 64, pass = 1;
  walk_row_tiles(lds, t, [&](RowTile& w) {
    if (rest || tiles <= wgs) return false;
    if (i == 64) {
      const int mine = shares.walked_entry(worker, pass + (int)(threadIdx.x & 63));   // (at most 2^31 tiles in all)
      const bool live = mine < shares.walked;
      int start, len, t, tm, tn;
      groups.find_lanes(p, live ? xcd * per_xcd + mine : 0, live, b.group, start, len, t);
      b.stream = local_tile(t, len > 0 ? (len + BM - 1) / BM : 1, (p.N + BN - 1) / BN, tm, tn) == 1;
      b.row = start + tm * BM;
      b.m_rem = len - tm * BM;
      b.col = tn * BN;
      b.count = __popcll(__ballot(live));
      pass += 64;
      i = 0;
    }
    if (i >= b.count) return false;
    tile_at(__builtin_amdgcn_readlane(b.group, i), __builtin_amdgcn_readlane(b.row, i), __builtin_amdgcn_readlane(b.m_rem, i),
            __builtin_amdgcn_readlane(b.col, i), __builtin_amdgcn_readlane(b.stream, i), w);
    ++i;
    return true;
  });
}

template <int LAYOUT, int BM, int BN, int BIAS>
__global__ __launch_bounds__(256) void grouped_device_kernel(DeviceGroups p) {
  using TS = TileShape<BM, BN>;
  __shared__ __attribute__((aligned(1024))) char lds[TS::LDS_BYTES];
  int t = blockIdx.x;
  if constexpr (LAYOUT == kGroupsUniform || LAYOUT == kGroupsPrepadM) {
    // The tile count is known on the host: XCD x works on a contiguous slice of the tile list.
    const int total = p.G * ((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN);
    const int per_xcd = (total + kXcds - 1) / kXcds;
    t = (blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
    if (t >= total) return;
  }
  GroupSpan sp;
  if (!find_group<LAYOUT, BM, BN>(p, t, sp)) return;
  const int64_t g = sp.gi, M = p.M, N = p.N, K = p.K;
  const int Mg = (LAYOUT == kGroupsSizesM || LAYOUT == kGroupsOffsetsM || LAYOUT == kGroupsPrepadM) ? sp.len : p.M;
  const int Ng = LAYOUT == kGroupsOffsetsN ? sp.len : p.N;
  const int Kg = LAYOUT == kGroupsOffsetsK ? sp.len : p.K;
  int tm, tn;
  local_tile(sp.t, ((LAYOUT == kGroupsPrepadM ? p.M : Mg) + BM - 1) / BM, (Ng + BN - 1) / BN, tm, tn);
  const int64_t m0 = tm * BM, n0 = tn * BN;
  if constexpr (LAYOUT == kGroupsPrepadM) {
    if (m0 >= sp.len) return;   // tile of padding rows only
  }
  const uint8_t *a, *b;
  const float *xs, *ws;
  uint16_t* y;
  if constexpr (LAYOUT == kGroupsSizesM || LAYOUT == kGroupsOffsetsM) {
    a = p.xq + (sp.o0 + m0) * K;      b = p.wq + (g * N + n0) * K;
    xs = p.xs + sp.o0 + m0;           ws = p.ws + g * N + n0;
    y = p.y + (sp.o0 + m0) * N + n0;
  } else if constexpr (LAYOUT == kGroupsOffsetsN) {
    a = p.xq + (g * M + m0) * K;      b = p.wq + (sp.o0 + n0) * K;
    xs = p.xs + g * M + m0;           ws = p.ws + sp.o0 + n0;
    y = p.y + m0 * N + sp.o0 + n0;
  } else if constexpr (LAYOUT == kGroupsOffsetsK) {
    a = p.xq + m0 * K + sp.o0;        b = p.wq + n0 * K + sp.o0;
    xs = p.xs + g * M + m0;           ws = p.ws + g * N + n0;
    y = p.y + (g * M + m0) * N + n0;
  } else {
    a = p.xq + (g * M + m0) * K;      b = p.wq + (g * N + n0) * K;
    xs = p.xs + g * M + m0;           ws = p.ws + g * N + n0;
    y = p.y + (g * M + m0) * N + n0;
  }
  const int m_rem = Mg - (int)m0, n_rem = Ng - (int)n0;
  const void* bias = nullptr;
  if constexpr (BIAS == 1) bias = static_cast<const float*>(p.bias) + g * N + n0;
  if constexpr (BIAS == 2) bias = static_cast<const uint16_t*>(p.bias) + g * N + n0;
  bool slow = p.unaligned != 0;
  if constexpr (LAYOUT == kGroupsOffsetsK) slow = slow || (sp.o0 & 15) != 0 || (Kg & 15) != 0;
  if (slow) {   // Kg == 0 needs no special case on either path: the sum is empty
    slow_tile<BM, BN, BIAS>(a, b, xs, ws, bias, y, m_rem, n_rem, p.N, Kg, K);
    return;
  }
  // A weight block that a single row tile reads at a time (the tile is the only one of its panel with rows to compute:
  // a group of at most BM rows, or the last panel of a group of 4 k + 1 row tiles) is fetched with non-temporal loads
  // (cfg4 307 -> 298 us, four big experts + eight of 256 rows 276 -> 253 us; with panels of two row tiles included:
  // cfg4 304 -> 315 us, a uniform batch of 512-row groups 268 -> 263 us -- not taken).
  const int live_tiles = (Mg + BM - 1) / BM, panel_first = tm / kGroupM * kGroupM;
  if (live_tiles - panel_first == 1) {
    GemmTile<TS, BIAS, false, true, TS::LA / 2, false, true> tile;
    tile.run(lds, a, b, xs, ws, bias, y, m_rem, n_rem, p.N, Kg, (uint32_t)p.K);
  } else {
    GemmTile<TS, BIAS, false, true> tile;
    tile.run(lds, a, b, xs, ws, bias, y, m_rem, n_rem, p.N, Kg, (uint32_t)p.K);
  }
}

template <int LAYOUT, int BM, int BN, int BIAS>
hipError_t launch_device_shape(const DeviceGroups& p, hipStream_t s) {
  const int64_t tiles_m = (p.M + BM - 1) / BM, tiles_n = (p.N + BN - 1) / BN;
  int64_t grid;
  if (LAYOUT == kGroupsOffsetsK) {
    // k_slice_tile(): whole runs for every XCD, which is no less than an eighth of the list for each
    const int64_t per = tiles_m * tiles_n, run = per > kXcds ? (per + kXcds - 1) / kXcds : 1;
    grid = ((p.G * per + run - 1) / run + kXcds - 1) / kXcds * kXcds * run;
  } else if (LAYOUT == kGroupsUniform || LAYOUT == kGroupsPrepadM) {
    grid = (p.G * tiles_m * tiles_n + kXcds - 1) / kXcds * kXcds;
  } else if (LAYOUT == kGroupsOffsetsN) {
    grid = (tiles_m * (tiles_n + p.G) + kXcds - 1) / kXcds * kXcds;   // every group may end in a partial tile; 8 slices
  } else {
    grid = ((tiles_m + p.G) * tiles_n + kXcds - 1) / kXcds * kXcds;
  }
  if (grid <= 0) return hipSuccess;
  if (grid > 2147483647) return hipErrorInvalidValue;
  if (dispatch_probe_record("grouped_device<%d,%d>%s workgroups=%lld", BM, BN, p.unaligned ? " unaligned" : "", (long long)grid)) return hipSuccess;
  grouped_device_kernel<LAYOUT, BM, BN, BIAS><<<(unsigned)grid, 256, 0, s>>>(p);
  return hipGetLastError();
}

// 128 x 128 or 256 x 256 tiles for groups of rows (sizes known on the host or not).  Two 128 x 128 workgroups share a CU, so
// one hides the other's first round trip and its epilogue; a 256 x 256 tile reads half as many operand bytes per product, and
// a ragged one costs what its rows cost.  The figures here are of sizes that fall like 1 / rank^1.1 and of weights that are not
// in the caches; equal sizes differ where tiles fill (launch_device_layout below).  The small tiles win where they all run at once (8 experts x 1536 x 2048 over 4096
// rows, 432 tiles: 19.8 against 27.5 us; 1 x 8192 x 5120 over 1024, 512 tiles: 47.0 / 54.4; but 2 x 4096 x 4096 over 2048, 544
// tiles: 52.4 / 43.1; 8 x 4096 x 2048 over 2048, 640 tiles: 37.9 / 27.0) and up to 128 rows per group, where the weight
// stream is the bound and half the rows of a 256-row tile are padding (64 x 2048 x 2048, by rows per group: 64 60.2 / 75.7,
// 128 78.6 / 78.4, 192 98.8 / 87.4, 256 110.5 / 104.7, 320 129.9 / 116.1; 16 x 4096 x 5120: 64 93.6 / 106.3, 128 107.4 /
// 109.4, 192 116.9 / 111.2, 320 156.2 / 124.8).  256 x 128 tiles were slower than either, 128 x 256 ones 5 % faster than
// 128 x 128 for few rows and K >= 4096 and slower otherwise.
// (Twice or four times the workgroups: not beyond kMaxWorkgroups, past which HIP refuses a launch that the larger tiles fit.)
constexpr int64_t kMaxWorkgroups = (int64_t(1) << 24) - 1;   // 256 lanes each, 2^32 work-items
inline bool small_row_groups(int64_t rows, int64_t groups, int64_t tiles128) {
  return rows <= 128 * groups || tiles128 <= 2 * device_compute_units();
}

template <int LAYOUT, int BIAS>
hipError_t launch_device_layout(const DeviceGroups& p, hipStream_t s) {
  const int64_t G = p.G > 0 ? p.G : 1;
  if constexpr (LAYOUT == kGroupsSizesM || LAYOUT == kGroupsOffsetsM) {
    // The sizes are not known here: a group ends in half a tile on average.  Where they may instead fill their tiles and those all
    // run at once (equal groups of a multiple of 128 rows), the small tiles win by a third and lose a fifth when the sizes are
    // skewed after all (8 x 4096 x 4096 over 2048 rows: equal 32 / 46 us, sizes like 1 / rank^1.1 59 / 48): the large ones are
    // taken, except for short K, where the small ones win or tie either way (8 x 1024 x 512 over 8192: 8.5 / 11.9 and 12.0 / 13.7;
    // 8 x 2048 x 768 over 4096: 10.1 / 14.0 and 14.8 / 15.7, but 16 of them 18.9 / 16.0).  Operands that take the scalar tile want many
    // workgroups (8 experts x 4096 x 1000 over 4096 rows: 32.0 ms, with 256 x 256 tiles 67.7).
    const int64_t M = p.M, N = p.N, tiles_m = G == 1 ? (M + 127) / 128 : (M + 64 * G) / 128, tiles128 = tiles_m * ((N + 127) / 128);
    const bool launchable = ((M + 127) / 128 + G) * ((N + 127) / 128) + kXcds <= kMaxWorkgroups;
    const int64_t full_tiles128 = ((M + 127) / 128) * ((N + 127) / 128);
    const bool short_k = p.K < 768 && full_tiles128 <= 2 * device_compute_units();
    if (launchable && (p.unaligned || short_k || small_row_groups(M, G, tiles128))) return launch_device_shape<LAYOUT, 128, 128, BIAS>(p, s);
    // The chain where there may be more tiles than CUs.  Without a second tile it has nothing to put a tile's end under, and its workgroups
    // of left-over tiles cost a launch each (K = 384 ... 2048 x 4096: one group of 4096 rows 8 - 17 % more than tiles one per
    // workgroup, two of 1024 16 %).
    const int64_t cus = device_compute_units();
    const int64_t most_tiles = (M + 255 * G) / 256 * ((N + 255) / 256);   // every group may end in a tile of one row
    if (!p.unaligned && M > 0 && most_tiles > cus && most_tiles <= 2147483647 && chain_takes(N, p.K, p.xq, p.wq, p.ws, p.y)) {
      if (dispatch_probe_record("grouped_rows<%d,%d> workgroups=%lld", RowTileShape::kBM, RowTileShape::kBN, (long long)(2 * cus))) return hipSuccess;
      grouped_rows_kernel<LAYOUT><<<(unsigned)(2 * cus), 256, 0, s>>>(p, (int)cus / kXcds);
      return hipGetLastError();
    }
    return launch_device_shape<LAYOUT, 256, 256, BIAS>(p, s);
  } else {
  // Tile shape from the average group: 256 x 256 once such tiles give every CU work.
  const int64_t Mg = p.M, Ng = LAYOUT == kGroupsOffsetsN ? (p.N + G - 1) / G : p.N;
  const int64_t big = G * ((Mg + 255) / 256) * ((Ng + 255) / 256);
  const int64_t pad = ((Mg + 255) / 256 * 256) * ((Ng + 255) / 256 * 256);
  const bool use_big = big >= 192 && pad * 4 <= Mg * Ng * 5;   // at most 25 % padding
  if (use_big) return launch_device_shape<LAYOUT, 256, 256, BIAS>(p, s);
  return launch_device_shape<LAYOUT, 128, 128, BIAS>(p, s);
  }
}

}  // namespace
}  // namespace mslk_amd
