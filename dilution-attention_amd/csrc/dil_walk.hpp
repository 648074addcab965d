// The row-parallel and key-parallel passes for calls that leave the chip idle:
// one 32-row (or 32-key) tile per workgroup, its walk split over the 4 waves.
//
// The full-chip forms (dil_forward_impl.hpp, dil_backward_impl.hpp) give a wave a
// tile of its own and stage the other side's tiles for 4 waves at once, which
// reads each tile once per 128 rows; a call then has slices * T / 128 workgroups
// and lasts as long as its longest wave: T / 32 tiles one after the other, 0.4 to
// 3 us each.  With few slices of short rows most of the chip has nothing to do
// meanwhile.  Here wave w of 4 takes every fourth tile of the walk (a quarter of
// the walk, for the demand), with its operands straight from L2 to registers, one
// tile ahead, and no barrier until the waves' sums are added: four times the
// workgroups, a quarter of the chain.  What it costs is the shared staging (four
// times the tile reads), so a full chip keeps the other forms (split_walks).
//
// The production operator only (softmax bids, dilution share).  All sums stay in
// fp32 (the demand's in fp64); only their order changes.
#pragma once

#include "dil_common.hpp"
#include "dil_internal.hpp"
#include "dil_tiles.hpp"

namespace dil {

namespace {

constexpr int kSplitWaves = 4;

// Whether the passes over `tiles` 32-row (or 32-key) tiles per slice split their
// walks.  The limits are where the two forms cross on 256 CUs; they fall with the
// operand bytes and registers of a tile and rise where a tile's products are
// slow.  Statistics + demand + output + dk correction, us, full-chip form -> split:
//   bf16 64:  64 tiles 59 -> 38, 645 tiles 121 -> 84, 1024 163 -> 136,
//            1280 193 -> 159, 1536 170 -> 183, 2048 (64 slices) 108 -> 145
//   bf16 32:  1024 tiles 145 -> 76, 2048 155 -> 128, 4096 265 -> 293 (no dk)
//   bf16 128: 504 tiles 220 -> 145, 756 221 -> 205, 1024 228 -> 257
//   fp32 64:  1024 tiles 593 -> 414, 1536 741 -> 612, 2048 793 -> 790, 4096 1178 -> 1549
//   fp32 128: 1024 tiles 1051 -> 850, 1536 1244 -> 1218, 2048 1347 -> 1607
//   split 64: 250 tiles 142 -> 83, 768 253 -> 232, 1024 256 -> 278, 1536 271 -> 403
//   split 32: 1024 tiles 189 -> 155, 1536 192 -> 199
//   split 128: 504 tiles 396 -> 301, 640 401 -> 376, 768 404 -> 422
template <typename CT, int D>
inline bool split_walks(int64_t n, int64_t tiles) {
  constexpr int64_t kLimit = std::is_same_v<CT, float>     ? (D <= 64 ? 2048 : 1024)
                             : std::is_same_v<CT, split32> ? (D <= 32 ? 1024 : 640)
                                                           : (D <= 32 ? 2048 : D <= 64 ? 1280 : 768);
  return n * tiles <= kLimit;
}

// Operand fragments straight from global memory, the layouts of lds_row_frag and
// lds_t_frag / lds_tq_frag.  Rows past the slice read its last row (their scores
// are masked); the tile-major transposes are padded with zeros.
template <typename CT, int D>
__device__ __forceinline__ void global_row_frag(RowFrag<CT, D>& f, const CT* base, int row, int last, int64_t ld, int h) {
  load_row_frag<CT, D>(f, base + min(row, last) * ld + h * (D / 2));
}

// The k slots of head dim r of a tile-major transpose's 32-row tile: QS false, in
// the permuted order (16 s + 8 h + [0, 8)); true, in the query-split order
// (16 h + 8 s + [0, 8)).
template <typename CT> constexpr int kSlots = kTileK / Mma<CT>::kStep;
template <typename CT, int D, bool QS>
__device__ __forceinline__ void global_t_frags(typename Mma<CT>::frag (&f)[kSlots<CT>], const CT* tile, int r, int h) {
  if (D < 32 && r >= D) {
#pragma unroll
    for (int s = 0; s < kSlots<CT>; ++s) f[s] = typename Mma<CT>::frag{};
    return;
  }
  const CT* row = tile + r * kTileK;
  if constexpr (kWideFrag<CT>) {
#pragma unroll
    for (int s = 0; s < kSlots<CT>; ++s) f[s] = frag8_at<CT>(row + (QS ? 16 * h + 8 * s : 16 * s + 8 * h));
  } else {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      // slots 4 u .. 4 u + 3: perm_row(s, h) = 16 (s >> 3) + 8 h + (s & 7), or 16 h + s
      const int at = QS ? 16 * h + 4 * u : 16 * (u >> 1) + 8 * h + 4 * (u & 1);
      const floatx4 x = *reinterpret_cast<const floatx4*>(row + at);
      f[4 * u] = x[0];
      f[4 * u + 1] = x[1];
      f[4 * u + 2] = x[2];
      f[4 * u + 3] = x[3];
    }
  }
}

// One tile's operands of a walk: the rows, and the transposed rows.
template <typename CT, int D, bool T>
struct WalkFrags {
  RowFrag<CT, D> row;
  typename Mma<CT>::frag t[T ? kDTiles<D> : 1][kSlots<CT>];
};

// The next tile's operands are loaded a step ahead where they fit the registers.
template <typename CT, int D>
constexpr bool kWalkAhead = D * sizeof(CT) <= 256;

// A wave's walk over tiles first, first + 4, ... < end: load(frags, tile) ahead,
// step(frags, tile).
template <bool AHEAD, typename F, typename L, typename S>
__device__ __forceinline__ void walk_tiles(int first, int end, L&& load, S&& step) {
  if constexpr (AHEAD) {
    F f[2];
    if (first < end) load(f[0], first);
    for (int kt = first; kt < end; kt += 2 * kSplitWaves) {
      if (kt + kSplitWaves < end) load(f[1], kt + kSplitWaves);
      step(f[0], kt);
      if (kt + kSplitWaves < end) {
        if (kt + 2 * kSplitWaves < end) load(f[0], kt + 2 * kSplitWaves);
        step(f[1], kt + kSplitWaves);
      }
    }
  } else {
    F f;
    for (int kt = first; kt < end; kt += kSplitWaves) {
      load(f, kt);
      step(f, kt);
    }
  }
}

}  // namespace
}  // namespace dil
