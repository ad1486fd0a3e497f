// Channel bias + GELU(tanh) fused with NCHW -> NHWC (channels-last), bf16.
//
// Semantics (the eager op order of gelu(x + bias) on bf16 tensors):
//   t = bf16(x + bias[c])            (fp32 add, round to nearest even)
//   y = bf16(GELU_tanh(t))           (fp32 arithmetic, one rounding)
// GELU_tanh(t) = 0.5 t (1 + tanh(u)), u = sqrt(2/pi) (t + 0.044715 t^3).
// t is a bf16 value, so the output is a function of its 65536 bit patterns,
// and the kernel returns the correctly rounded bf16 of the exact function
// (gelu_bf16.h: an fp32 evaluation for t > -4 that rounds correctly for
// every such bf16 t, the exact table in global memory below that).
//
// Layout: 8 x 8 (channel x position) register blocks, 64 of them to a wave
// (block_tiles.h): 8 16-byte loads along the channel rows, 8 16-byte stores
// along the NHWC rows, the transpose in registers, with no LDS and no
// barrier (a 7 KiB table staged into LDS by every workgroup cost 3-5 us at
// [128, 256, 56, 56]).  Channel tiles are numbered fastest, so a workgroup's
// four waves write neighbouring parts of the same NHWC rows.  The grid is
// one-shot (a persistent one-workgroup-per-CU version ran 71 us there).
// Planes and channel counts of any size >= 8 take it; before, those that are
// not multiples of 8 took the one-element-per-thread kernel.  Graph replays,
// before -> now: [128, 384, 14, 14] 49.2 -> 9.4 us, [128, 1024, 14, 14] 111
// -> 18, [128, 512, 7, 7] 15.3 -> 5.4, [13, 230, 77, 74] 82 -> 14.6; and,
// multiples of 8, [128, 512, 28, 28] 49.8 -> 38.7, [128, 256, 28, 28] 27.6 ->
// 17.8, [128, 16, 112, 112] 48 -> 20 ([128, 256, 56, 56] 70 either way).  What is left at 14 x 14
// (floor 5.8 us) is arithmetic: about 23 issue slots per value.
// Launches of at most 2^19 elements, and images of few values, take the
// one-element-per-thread kernel.
// HBM-bound: algorithmic bytes per element = 2 (read) + 2 (write).
#include "block_tiles.h"
#include "gelu_bf16.h"

namespace hipo {
namespace {

constexpr int64_t kTileMinElems = int64_t{1} << 19;  // smaller launches: scalar kernel

template <TileAccess ACCESS>
__global__ __launch_bounds__(kTileThreads) void bias_gelu_nchw_to_nhwc_blocks(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ bias,
    uint16_t* __restrict__ out, BlockTiles t) {
  const BlockPlace p = block_place(t, 8);  // t.R channels, t.C positions
  const int64_t img = static_cast<int64_t>(p.mat) * t.R * t.C;
  const uint16_t* xb = x + img + p.r * t.C + p.c;
  u32x4_t v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = tile_load<ACCESS>(xb + j * t.C);
  const u32x4_t bw = *reinterpret_cast<const u32x4_a2_t*>(bias + p.r);
  float b[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) b[j] = (j & 1) ? bf16hi(bw[j >> 1]) : bf16lo(bw[j >> 1]);
  if (!p.own) return;  // no barrier follows
  uint16_t* ob = out + img + p.c * t.R + p.r;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    // Position p.c + i, channels p.r .. p.r + 7: round t for two channels
    // into one word (v_cvt_pk_bf16_f32), map both halves, pack them.
    u32x4_t o, tt;
    bool rare = false;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t w0 = v[2 * k][i >> 1];
      const uint32_t w1 = v[2 * k + 1][i >> 1];
      const float x0 = (i & 1) ? bf16hi(w0) : bf16lo(w0);
      const float x1 = (i & 1) ? bf16hi(w1) : bf16lo(w1);
      tt[k] = pack_bf16x2(x0 + b[2 * k], x1 + b[2 * k + 1]);
      o[k] = gelu_pair_fast(tt[k], rare);
    }
    if (rare) {  // one branch per 8 values, rarely taken for ordinary data
      gelu_exact_x8(tt, o);
    }
    tile_store<ACCESS>(o, ob + i * t.R);
  }
}

// Any shape: one thread per output element, NHWC order (coalesced stores,
// strided loads); the same mapping as the tile kernel, from the table in
// global memory.
__global__ __launch_bounds__(256) void bias_gelu_nchw_to_nhwc_scalar(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ bias,
    uint16_t* __restrict__ out, int64_t N, int64_t C, int64_t HW) {
  const int64_t total = N * C * HW;
  for (int64_t o = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
       o < total; o += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t c = o % C;
    const int64_t p = (o / C) % HW;
    const int64_t img = o / (C * HW);
    const uint32_t tb =
        pack_bf16x2(bf16_to_f32(x[(img * C + c) * HW + p]) + bf16_to_f32(bias[c]), 0.0f) &
        0xffffu;
    out[o] = static_cast<uint16_t>(gelu_bits(tb, kGeluTable));
  }
}

// Whether the tiles beat a thread per element.  A wave maps 64 values a lane
// one after the other, however few of its lanes own a block and however much
// the last blocks overlap; a thread per element reads a cache line for each of
// its wave's channels, which longer planes of many channels do not find in the
// L1 again for their next positions.  Estimates in us of both, fitted to graph
// replays over 9 to 1500 channels, planes of 9 to 1369 positions and 0.55 to 8
// million elements: of 1499 points 18 come out over 5 % slower than the better of
// the two, the worst 18 %.  Measured, tiles / thread per element: [60000, 9, 3, 3]
// 91 / 18, [64, 1000, 3, 3] 8.2 / 4.2, [3000, 64, 2, 5] 10.6 / 8.8, [2187, 16, 4, 4]
// 10.6 / 4.2, [9375, 64, 3, 5] 25 / 30, [834, 40, 6, 6] 5.0 / 5.8, [128, 512, 7, 7]
// 8.7 / 16.3, [19, 640, 12, 9] 5.1 / 9.4, [2, 982, 19, 21] 4.6 / 5.6.  Images of whole
// blocks keep the tiles from kTileMinElems on unless their waves alone cost more.
bool tiles_pay(const BlockTiles& t, int64_t elements, int64_t c, int64_t hw, bool whole) {
  const auto ramp = [](int64_t v, double from, double to) {
    return std::min(1.0, std::max(0.0, (static_cast<double>(v) - from) / (to - from)));
  };
  const double element_us = 3.05e-6 * (1.0 + 0.6 * ramp(hw, 20, 60) * ramp(c, 60, 260));
  const double tiles_us = whole ? 1.7e-3 * t.waves : 2.8 + 1.3e-3 * t.waves;
  return tiles_us < element_us * static_cast<double>(elements);
}

}  // namespace
}  // namespace hipo

extern "C" int hipo_bias_gelu_nchw_to_nhwc_bf16(const uint16_t* x,
                                                const uint16_t* bias,
                                                uint16_t* out, int64_t n,
                                                int64_t c, int64_t hw,
                                                hipStream_t stream) {
  using namespace hipo;
  clear_error();
  HIPO_REQUIRE(n >= 0 && c >= 0 && hw >= 0, "bias_gelu: negative size");
  if (n == 0 || c == 0 || hw == 0) return 0;
  HIPO_REQUIRE(x && bias && out, "bias_gelu: null pointer");
  // Up to kTileMinElems elements the one-element-per-thread kernel is the
  // faster one: a tile wave maps its 4096 values serially (64 per lane), so
  // a launch of few tiles is bound by one wave's instruction stream, not by
  // memory (steady-state: 5.4 against 2.5 us at [3, 320, 8, 10], 5.9
  // against 3.2 us at [4, 128, 28, 28]; 6.7 against 10.8 us at
  // [2, 256, 56, 56], where the tiles win).
  BlockTiles t;
  TileAccess access;
  const bool whole = c % 8 == 0 && hw % 8 == 0 && aligned16(x) && aligned16(out);
  if (n * c * hw > kTileMinElems && block_tiles(x, out, n, c, hw, 2, t, access) &&
      tiles_pay(t, n * c * hw, c, hw, whole)) {
    auto kernel = access == TileAccess::kCached
                      ? bias_gelu_nchw_to_nhwc_blocks<TileAccess::kCached>
                  : access == TileAccess::kStreamOut
                      ? bias_gelu_nchw_to_nhwc_blocks<TileAccess::kStreamOut>
                      : bias_gelu_nchw_to_nhwc_blocks<TileAccess::kStream>;
    kernel<<<dim3(t.workgroups()), dim3(kTileThreads), 0, stream>>>(x, bias, out, t);
  } else {
    const int64_t total = n * c * hw;
    int64_t blocks = (total + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    bias_gelu_nchw_to_nhwc_scalar<<<dim3(static_cast<unsigned>(blocks)),
                                    dim3(256), 0, stream>>>(x, bias, out, n, c,
                                                            hw);
  }
  return check_launch("bias_gelu_nchw_to_nhwc_bf16");
}
