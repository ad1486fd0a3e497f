// Work layout of the transposing kernels: [R, C] matrices, `mats` of them,
// written as [C, R].
//
// A lane owns a V x V block (V = 16 bytes of elements): V 16-byte loads, one
// per row, and, after a transpose in registers, V 16-byte stores, one per
// column.  A wave's lanes hold br x bc blocks, lane = (block row) * bc +
// (block column), so a load instruction reads br runs of 16 * bc contiguous
// bytes and a store instruction writes bc runs of 16 * br.  Blocks that would
// cross the end of the rows or columns move back to end there; what they
// share with their neighbour both store with the same bytes.  No LDS, no
// barrier.
//
// Waves are numbered row tile fastest, then column tile, then matrix, four
// consecutive ones to a workgroup, workgroups in XCD order: tiles that share
// cache lines (rows that are not whole lines share one at every tile edge)
// run close together on one L2.
//
// Cache policy (TileAccess).  Output rows that share 16-byte vectors, or
// shorter than a cache line: cached loads and stores, so that the pieces of
// a line meet in the L2.  Else, up to 160 MB read and written: cached loads,
// non-temporal stores, which leave the Infinity Cache to an input that is read
// again (one read for the first time, or just produced, is read faster by
// non-temporal loads: each of 1.2 GB of inputs transposed behind the
// elementwise kernel that wrote it, [24, 1024, 768] 14.1 us this way, 12.8 that;
// [40, 512, 512] 8.4, 8.0).  Beyond: non-temporal both ways where all rows are whole
// cache lines (in plain order where a workgroup's four tiles cover the
// output rows), cached both ways otherwise; up to 32 MB of whole lines
// non-temporal both ways too.  Graph replays in us, cached /
// cached loads only / non-temporal, all in XCD order, then non-temporal in
// plain order; three inputs and one output reused, and in brackets 1.2 GB of
// inputs and outputs in turn:
//   transpose [24, 1024, 768] bf16, 75 MB   14.4 / 12.6 / 16.6 / 15.6  [20.3 18.3 17.6 16.5]
//   transpose [120, 1024, 768] bf16         74.3 / 68.3 / 65.9 / 72.5  [74.2 68.3 66.2 72.3]
//   transpose [192, 1024, 768] bf16         114 / 107 / 103 / 117      [113 107 103 117]
//   transpose [128, 197, 768] bf16          16.7 / 22 / 22 / 23        [22.8 34.3 33.1 33.6]
//   transpose [128, 768, 197] bf16          13.9 / - / - / -           [21.1 21.2 21.6 24.3]
//   bias_gelu [8, 256, 56, 56], 26 MB       8.6 / 7.3 / 6.8 / 7.0      [10.1 8.7 8.3 8.2]
//   bias_gelu [128, 384, 14, 14]            - / 9.4 / - / 15.2         [13.8 14.0 14.0 15.6]
//   bias_gelu [64, 256, 56, 56], 205 MB     34.4 / 40.4 / 39.5 / 37.0  [42.1 39.6 39.5 37.1]
//   bias_gelu [128, 256, 56, 56]            79.1 / 76.8 / 75.0 / 69.8  [76.7 75.2 73.7 68.2]
//   bias_gelu [128, 512, 28, 28], 205 MB    38.7 / 42.7 / 45.6 / 49.8  [42.6 41.7 43.9 49.1]
//   bias_gelu [128, 16, 112, 112]           19.9 / 53.3 / - / 54       [30.2 59.8 55.2 50.4]
//
// Shape of a wave's tile: 8 x 8 blocks, unless the matrix divides badly into
// those and another br x bc <= 64 leaves over 5 % fewer lanes idle (25 x 96
// blocks: 5 x 12 uses 94 % of the lanes, 8 x 8 78 %).  Runs stay at least 64
// bytes where the matrix has them.
#pragma once

#include <algorithm>

#include "hipo_common.h"

namespace hipo {

constexpr int kTileWaves = 4;  // per workgroup
constexpr int kTileThreads = kTileWaves * kWave;

enum class TileAccess { kCached, kStreamOut, kStream };
constexpr int64_t kTileSmallBytes = 32'000'000;   // read and written together
constexpr int64_t kTileCacheBytes = 160'000'000;

// 16 bytes at any element's address.
template <TileAccess ACCESS>
__device__ __forceinline__ u32x4_t tile_load(const void* p) {
  const u32x4_a2_t* v = static_cast<const u32x4_a2_t*>(p);
  return ACCESS == TileAccess::kStream ? __builtin_nontemporal_load(v) : *v;
}

template <TileAccess ACCESS>
__device__ __forceinline__ void tile_store(u32x4_t v, void* p) {
  u32x4_a2_t* d = static_cast<u32x4_a2_t*>(p);
  if constexpr (ACCESS != TileAccess::kCached) {
    __builtin_nontemporal_store(v, d);
  } else {
    *d = v;
  }
}

struct BlockTiles {
  int64_t R, C;
  uint32_t waves;           // tiles in all: rtiles * ctiles * mats < 2^31
  uint32_t rtiles, ctiles;  // tiles of one matrix
  uint32_t br, bc;          // blocks per tile
  uint32_t lane_magic;      // lane / bc == (lane * lane_magic) >> 16
  DivMagic by_rtiles, by_ctiles;
  uint32_t plain_order;     // 1: workgroups in launch order
  unsigned workgroups() const { return (waves + kTileWaves - 1) / kTileWaves; }
};

// Lanes of a br x bc tile that own a block, of all lanes of all tiles.
inline double tile_use(int64_t RB, int64_t CB, int64_t br, int64_t bc) {
  const int64_t tiles = (RB + br - 1) / br * ((CB + bc - 1) / bc);
  return static_cast<double>(RB * CB) / static_cast<double>(tiles * kWave);
}

// The tiles of `mats` [R, C] matrices of `size`-byte elements at x, written
// as [C, R] at y, and their cache policy.  False: R or C below one block, or
// too many tiles for the 32-bit index.
inline bool block_tiles(const void* x, const void* y, int64_t mats, int64_t R, int64_t C,
                        int size, BlockTiles& t, TileAccess& access) {
  const int V = 16 / size;
  if (R < V || C < V) return false;
  const int64_t RB = (R + V - 1) / V, CB = (C + V - 1) / V;
  int64_t br = 8, bc = 8;
  double best = 1.05 * tile_use(RB, CB, br, bc);
  for (int64_t b = std::min<int64_t>(4, CB); b <= std::min<int64_t>(kWave, CB); ++b) {
    const int64_t a = std::min<int64_t>(kWave / b, RB);
    if (a < std::min<int64_t>(4, RB)) break;
    const double use = tile_use(RB, CB, a, b);
    if (use > best) best = use, br = a, bc = b;
  }
  const int64_t rtiles = (RB + br - 1) / br, ctiles = (CB + bc - 1) / bc;
  constexpr int64_t kMost = (int64_t{1} << 31) - kTileWaves;
  if (rtiles * ctiles >= kMost || mats >= kMost || rtiles * ctiles * mats >= kMost) return false;
  t.R = R;
  t.C = C;
  t.waves = static_cast<uint32_t>(rtiles * ctiles * mats);
  t.rtiles = static_cast<uint32_t>(rtiles);
  t.ctiles = static_cast<uint32_t>(ctiles);
  t.br = static_cast<uint32_t>(br);
  t.bc = static_cast<uint32_t>(bc);
  t.lane_magic = (0x10000u + t.bc - 1) / t.bc;
  t.by_rtiles = div_magic(t.rtiles);
  t.by_ctiles = div_magic(t.ctiles);
  t.plain_order = 0;
  const int64_t in_row = C * size, out_row = R * size;
  if (out_row % 16 != 0 || !aligned16(y) || out_row < 128) {
    access = TileAccess::kCached;
  } else {
    const int64_t bytes = 2 * mats * R * in_row;
    const bool lines = in_row % 128 == 0 && out_row % 128 == 0 && aligned16(x);
    if (lines && (bytes <= kTileSmallBytes || bytes > kTileCacheBytes)) {
      access = TileAccess::kStream;
    } else {
      access = bytes <= kTileCacheBytes ? TileAccess::kStreamOut : TileAccess::kCached;
    }
    if (access == TileAccess::kStream && bytes > kTileCacheBytes && rtiles <= kTileWaves)
      t.plain_order = 1;
  }
  return true;
}

// This lane's block: rows r .. r + V - 1, columns c .. c + V - 1 of matrix
// `mat`; `own` is false for a lane without one (its addresses are in bounds).
struct BlockPlace {
  uint32_t mat;
  int64_t r, c;
  bool own;
};

__device__ __forceinline__ BlockPlace block_place(const BlockTiles& t, int V) {
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t bid = t.plain_order ? blockIdx.x : xcd_order(blockIdx.x, gridDim.x);
  const uint32_t w0 = __builtin_amdgcn_readfirstlane(bid * kTileWaves + (threadIdx.x >> 6));
  const uint32_t w = w0 < t.waves ? w0 : t.waves - 1;
  const uint32_t rest = div_by(w, t.by_rtiles);
  const uint32_t rt = w - rest * t.rtiles;
  const uint32_t mat = div_by(rest, t.by_ctiles);
  const uint32_t ct = rest - mat * t.ctiles;
  const uint32_t ri = (lane * t.lane_magic) >> 16;
  const uint32_t ci = lane - ri * t.bc;
  const int64_t r = static_cast<int64_t>(rt * t.br + ri) * V;
  const int64_t c = static_cast<int64_t>(ct * t.bc + ci) * V;
  BlockPlace p;
  p.mat = mat;
  p.own = w0 < t.waves && ri < t.br && r < t.R && c < t.C;
  p.r = std::min<int64_t>(r, t.R - V);
  p.c = std::min<int64_t>(c, t.C - V);
  return p;
}

}  // namespace hipo
