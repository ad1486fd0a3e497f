// Row mean, fp32: out[r] = sum(x[r, :]) / cols.
//
// Several waves per row.  A workgroup holds `rows_per_block` rows of
// `waves_per_row` waves each (at most 8 waves).  Lane l of wave w of a row
// reads float4 index  (it * U + u) * W * 64 + w * 64 + l  (W = waves per
// row), so every load instruction of a wave covers 1 KiB of contiguous row
// and the W waves of a row sweep it together.  Each lane keeps U
// non-temporal 16-byte loads in flight, accumulates in fp32, the wave
// reduces with DPP, and the W wave sums are added in LDS in a fixed order.
//
// Measured on MI355X for [8192, 4096]: 8 waves x 2 float4 per lane reads at
// 81 % of 8 TB/s; one wave per row with 16 float4 per lane reaches 67 %
// (73 % with non-temporal loads) -- smaller per-wave footprints keep the
// in-flight address window compact.
// HBM-bound: algorithmic bytes per row = 4*cols (read) + 4 (write).
#include <algorithm>

#include "row_layout.h"

namespace hipo {
namespace {

constexpr int kMaxWaves = 8;  // per workgroup
constexpr int kMaxThreads = kMaxWaves * kWave;
constexpr int64_t kRaggedMinCols = 1024;
constexpr int64_t kRaggedMaxRows = 2048;

// WT > 0: waves per row (and rows per workgroup, kMaxWaves / WT) fixed at
// compile time; WT = 0: both from the arguments.
// RAGGED: rows of any length >= 4, any stride and alignment: a row's last
// float4 moves back to end with it, where its first values, its neighbour's,
// count as zero; loads at element alignment.
template <int U, int WT, bool RAGGED>
__global__ __launch_bounds__(kMaxThreads) void row_mean_f32_vec4(
    const float* __restrict__ x, float* __restrict__ out, int64_t rows,
    int64_t cols, int64_t row_stride, int w_arg, int rpb_arg) {
  const int waves_per_row = WT > 0 ? WT : w_arg;
  const int rows_per_block = WT > 0 ? kMaxWaves / WT : rpb_arg;
  __shared__ float part[kMaxWaves];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x >> 6;
  const int w = wave % waves_per_row;
  const int64_t row =
      static_cast<int64_t>(blockIdx.x) * rows_per_block + wave / waves_per_row;
  // Waves past the last row still take part in the barrier; they read the
  // last row and write nothing.
  const bool valid = row < rows;
  const float* xr = x + (valid ? row : rows - 1) * row_stride;
  const f32x4_t* p = reinterpret_cast<const f32x4_t*>(xr);
  const int64_t nvec = RAGGED ? (cols + 3) >> 2 : cols >> 2;
  const int64_t step = static_cast<int64_t>(waves_per_row) * kWave;

  const int64_t sweeps = (nvec + step * U - 1) / (step * U);

  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  for (int64_t it = 0; it < sweeps; ++it) {
    const int64_t base = it * step * U + w * kWave + lane;
    f32x4_t v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // Out-of-row slots load the row's last float4 (in bounds, no branch
      // around the load) and are zeroed.
      const int64_t i = base + u * step;
      if constexpr (RAGGED) {
        const int64_t at = i * 4 < cols - 4 ? i * 4 : cols - 4;
        const int64_t skip = i * 4 - at;  // >= 4: past the row
        v[u] = *reinterpret_cast<const f32x4_a4_t*>(xr + at);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[u][e] = e >= skip ? v[u][e] : 0.f;
      } else {
        v[u] = __builtin_nontemporal_load(p + (i < nvec ? i : nvec - 1));
        if (i >= nvec) v[u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) acc += v[u];
  }
  float s = wave_sum((acc.x + acc.y) + (acc.z + acc.w));
  if (waves_per_row > 1) {
    if (lane == 0) part[wave] = s;
    __syncthreads();
    const int first = wave - w;
    s = part[first];
    for (int k = 1; k < waves_per_row; ++k) s += part[first + k];
  }
  if (valid && w == 0 && lane == 0) out[row] = s / static_cast<float>(cols);
}

// Any alignment, any cols: scalar loads, one wave per row (many rows, or short
// ones; see the entry point).
__global__ __launch_bounds__(256) void row_mean_f32_scalar(
    const float* __restrict__ x, float* __restrict__ out, int64_t rows,
    int64_t cols, int64_t row_stride) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t row = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const float* p = x + row * row_stride;
  // Eight loads per lane in flight before any add (one at a time, every
  // iteration waited a full memory latency); the adds keep the order
  // i = lane, lane + 64, ... and skip what lies past the row, so the sum is
  // the same as a one-by-one loop's.
  constexpr int kBatch = 8;
  float acc = 0.f;
  for (int64_t i0 = lane; i0 < cols; i0 += int64_t{kWave} * kBatch) {
    float v[kBatch];
#pragma unroll
    for (int k = 0; k < kBatch; ++k) {
      const int64_t i = i0 + int64_t{k} * kWave;
      v[k] = i < cols ? p[i] : 0.f;
    }
#pragma unroll
    for (int k = 0; k < kBatch; ++k)
      if (i0 + int64_t{k} * kWave < cols) acc += v[k];
  }
  const float s = wave_sum(acc);
  if (lane == 0) out[row] = s / static_cast<float>(cols);
}


// bf16 rows, fp32 accumulation, optional ReLU (NaN kept):
//   out[r] = bf16(sum_j act(x[r, j]) / cols)   (one rounding, nearest even).
// Short rows (cols <= 512, contiguous): each wave takes 8
// consecutive rows -- 16 * cols bytes, a whole number of 16-byte vectors
// whatever cols is, so the input is read as one flat stream of non-temporal
// vector loads (the SqueezeNet rows are 169 elements, 338 bytes, not
// vector-aligned one by one), element-aligned ones (ALIGNED false) where x is
// off 16 bytes.  The wave stages its 8 rows in LDS; then 8
// lanes per row sum every 8th element in order and combine in a fixed
// DPP butterfly.
constexpr int kBf16RowsPerWave = 8;
constexpr int kBf16ShortCols = 512;
constexpr int kBf16Waves = 4;
constexpr int64_t kBf16ShortRows = 24000;  // from here on also off alignment

template <bool RELU>
__device__ __forceinline__ float act_relu(float v) {
  return RELU ? __builtin_elementwise_maximum(v, 0.0f) : v;
}

__device__ __forceinline__ uint16_t round_to_bf16(float v) {
  return static_cast<uint16_t>(pack_bf16x2(v, 0.0f) & 0xffffu);
}

template <bool RELU, int VPL, bool ALIGNED>
__global__ __launch_bounds__(kBf16Waves * kWave) void row_mean_bf16_short(
    const uint16_t* __restrict__ x, uint16_t* __restrict__ out, int64_t rows, int cols) {
  __shared__ __align__(16) uint16_t stage[kBf16Waves][kBf16RowsPerWave * kBf16ShortCols];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x >> 6;
  const int64_t row0 = (static_cast<int64_t>(blockIdx.x) * kBf16Waves + wave) * kBf16RowsPerWave;
  const int64_t nrows = rows - row0 < kBf16RowsPerWave ? rows - row0 : kBf16RowsPerWave;
  uint16_t* lds = stage[wave];
  if (nrows > 0) {
    // The wave's rows: `cols` vectors of 16 bytes when all 8 rows exist;
    // the last group may end inside a vector, whose elements move singly.
    const int64_t elems = nrows * cols;
    const int whole = static_cast<int>(elems / 8);
    const u32x4_t* xv = reinterpret_cast<const u32x4_t*>(x + row0 * cols);
    if (whole > 0) {  // wave-uniform
      // Loads without a branch (slots past the end reload the last vector),
      // so all of them are in flight before the first is used.
      u32x4_t v[VPL];
#pragma unroll
      for (int k = 0; k < VPL; ++k) {
        const int i = lane + k * kWave;
        if constexpr (ALIGNED) {
          v[k] = __builtin_nontemporal_load(xv + (i < whole ? i : whole - 1));
        } else {
          v[k] = ragged_load_stream(x + row0 * cols + (i < whole ? i : whole - 1) * 8);
        }
      }
#pragma unroll
      for (int k = 0; k < VPL; ++k) {
        const int i = lane + k * kWave;
        if (i < whole) reinterpret_cast<u32x4_t*>(lds)[i] = v[k];
      }
    }
    const int rest = static_cast<int>(elems - int64_t{whole} * 8);
    if (lane < rest) lds[whole * 8 + lane] = x[row0 * cols + whole * 8 + lane];
  }
  __syncthreads();
  if (nrows <= 0) return;
  const int r = lane >> 3;   // row of the group
  const int k = lane & 7;    // this lane's residue class
  float s = 0.0f;
  if (r < nrows) {
    const uint16_t* p = lds + r * cols;
    for (int j = k; j < cols; j += 8) s += act_relu<RELU>(bf16_to_f32(p[j]));
  }
  s = sum8(s);
  if (k == 0 && r < nrows) out[row0 + r] = round_to_bf16(s / static_cast<float>(cols));
}

// A wave per row, one load per lane in flight: many whole rows that would leave
// much of the kernel below's loads past their ends (VEC: 16-byte loads), and
// short ones off 16-byte alignment (single values); see the entry point.
template <bool RELU, bool VEC>
__global__ __launch_bounds__(kBf16Waves * kWave) void row_mean_bf16_wave(
    const uint16_t* __restrict__ x, uint16_t* __restrict__ out, int64_t rows, int64_t cols) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kBf16Waves + (threadIdx.x >> 6);
  if (row >= rows) return;  // wave-uniform; no barrier follows
  const uint16_t* xr = x + row * cols;
  float acc = 0.0f;
  if constexpr (VEC) {
    const u32x4_t* p = reinterpret_cast<const u32x4_t*>(xr);
    for (int64_t i = lane; i < cols / kRowGroup; i += kWave) {
      const u32x4_t v = __builtin_nontemporal_load(p + i);
      float t = 0.0f;
#pragma unroll
      for (int d = 0; d < 4; ++d)
        t += act_relu<RELU>(bf16lo(v[d])) + act_relu<RELU>(bf16hi(v[d]));
      acc += t;
    }
  } else {
    for (int64_t i = lane; i < cols; i += kWave) acc += act_relu<RELU>(bf16_to_f32(xr[i]));
  }
  const float s = wave_sum(acc);
  if (lane == 0) out[row] = round_to_bf16(s / static_cast<float>(cols));
}

// Longer rows: W waves per row as in row_mean_f32_vec4, U 16-byte loads per
// lane in flight; RAGGED: any length >= 8 and alignment, the row's last group
// moved back to end with it (RaggedGroup), element-aligned cached loads.
// Against one wave per row with one load in flight, graph replays: [2000, 16001]
// 74.5 -> 12.0 us, [20, 16000] 7.0 -> 3.0, [16000, 777] 10.7 -> 6.3, [8000, 4096]
// 11.7 -> 11.8.
template <bool RELU, int U, bool RAGGED>
__global__ __launch_bounds__(kMaxThreads) void row_mean_bf16_rows(
    const uint16_t* __restrict__ x, uint16_t* __restrict__ out, int64_t rows, int64_t cols,
    int waves_per_row, int rows_per_block) {
  __shared__ float part[kMaxWaves];
  const RowPlace p = row_place(waves_per_row, rows_per_block, rows);
  const uint16_t* xr = x + p.row * cols;
  const int64_t sweep = static_cast<int64_t>(waves_per_row) * kRowSweep;
  float acc = 0.0f;
  for (int64_t base = 0; base < cols; base += sweep * U) {
    u32x4_t v[U];
    int skip[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const RaggedGroup rg = ragged_group(base + row_group_col(u, waves_per_row, p), cols);
      v[u] = RAGGED ? ragged_load_cached(xr + rg.col)
                    : __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(xr + rg.col));
      skip[u] = rg.skip;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        acc += skip[u] <= 2 * d ? act_relu<RELU>(bf16lo(v[u][d])) : 0.0f;
        acc += skip[u] <= 2 * d + 1 ? act_relu<RELU>(bf16hi(v[u][d])) : 0.0f;
      }
    }
  }
  float s = wave_sum(acc);
  if (waves_per_row > 1) {
    if (p.lane == 0) part[p.wave] = s;
    __syncthreads();
    const int first = p.wave - p.w;
    s = part[first];
    for (int k = 1; k < waves_per_row; ++k) s += part[first + k];
  }
  if (p.valid && p.w == 0 && p.lane == 0) out[p.row] = round_to_bf16(s / static_cast<float>(cols));
}

// Fewer than 8 values off 16-byte alignment: a lane per row.
template <bool RELU>
__global__ __launch_bounds__(256) void row_mean_bf16_scalar(const uint16_t* __restrict__ x,
                                                            uint16_t* __restrict__ out,
                                                            int64_t rows, int64_t cols) {
  const int64_t row = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (row >= rows) return;
  float acc = 0.0f;
  for (int64_t i = 0; i < cols; ++i) acc += act_relu<RELU>(bf16_to_f32(x[row * cols + i]));
  out[row] = round_to_bf16(acc / static_cast<float>(cols));
}

}  // namespace
}  // namespace hipo

extern "C" int hipo_row_mean_f32(const float* x, float* out, int64_t rows,
                                 int64_t cols, int64_t row_stride,
                                 hipStream_t stream) {
  using namespace hipo;
  clear_error();
  HIPO_REQUIRE(rows >= 0 && cols >= 0, "row_mean: negative size");
  HIPO_REQUIRE(row_stride >= cols, "row_mean: row_stride %lld < cols %lld",
               (long long)row_stride, (long long)cols);
  if (rows == 0) return 0;
  HIPO_REQUIRE(x != nullptr && out != nullptr, "row_mean: null pointer");
  const bool vec = (cols % 4 == 0) && (row_stride % 4 == 0) && aligned16(x);
  // Rows off the vector path: one wave per row with 4-byte loads is as fast
  // where the rows alone fill the chip, and faster for short ones ([65536, 17]
  // 9.2 us against 11.2, [4000, 4097] 11.2 against 12.2); few long rows take
  // several waves each ([24, 8707] 7.2 -> 3.1 us, [1536, 1537] 4.3 -> 4.1, [1920,
  // 12001] 21.4 -> 16.4, but [2047, 1025] 3.6 -> 4.0, [1300, 1025] 3.4 -> 3.6).
  const bool ragged = !vec && rows < kRaggedMaxRows &&
                      cols >= (rows < kRaggedMaxRows / 2 ? kRaggedMinCols
                                                         : kRaggedMinCols * 3 / 2);
  if (cols >= 4 && (vec || ragged)) {
    // About 2 KiB per wave: W = ceil(nvec / 128) waves per row (at most 8),
    // U = float4 per lane per sweep.
    const int64_t nvec = (cols + 3) / 4;
    const int waves = static_cast<int>(
        std::min<int64_t>(kMaxWaves, (nvec + 2 * kWave - 1) / (2 * kWave)));
    const int64_t per_lane = (nvec + int64_t{waves} * kWave - 1) / (int64_t{waves} * kWave);
    const int rpb = kMaxWaves / waves;
    const int64_t blocks = (rows + rpb - 1) / rpb;
    HIPO_REQUIRE(blocks <= 0x7fffffff, "row_mean: too many rows");
    const dim3 grid(static_cast<unsigned>(blocks)), block(waves * rpb * kWave);
#define HIPO_MEAN(U_, W_)                                                            \
  row_mean_f32_vec4<U_, W_, false><<<grid, block, 0, stream>>>(x, out, rows, cols,   \
                                                               row_stride, waves, rpb)
#define HIPO_MEAN_RAGGED(U_)                                                         \
  row_mean_f32_vec4<U_, 0, true><<<grid, block, 0, stream>>>(x, out, rows, cols,     \
                                                             row_stride, waves, rpb)
#define HIPO_MEAN_W(U_)                                  \
  switch (waves) {                                       \
    case 1: HIPO_MEAN(U_, 1); break;                     \
    case 2: HIPO_MEAN(U_, 2); break;                     \
    case 4: HIPO_MEAN(U_, 4); break;                     \
    case 8: HIPO_MEAN(U_, 8); break;                     \
    default: HIPO_MEAN(U_, 0); break;                    \
  }
    if (!vec) {
      if (per_lane <= 1) HIPO_MEAN_RAGGED(1);
      else if (per_lane <= 2) HIPO_MEAN_RAGGED(2);
      else HIPO_MEAN_RAGGED(4);
    } else if (per_lane <= 1) {
      HIPO_MEAN_W(1);
    } else if (per_lane <= 2) {
      HIPO_MEAN_W(2);
    } else {
      HIPO_MEAN_W(4);
    }
#undef HIPO_MEAN_RAGGED
#undef HIPO_MEAN_W
#undef HIPO_MEAN
  } else {
    const int64_t blocks = (rows + 3) / 4;
    HIPO_REQUIRE(blocks <= 0x7fffffff, "row_mean: too many rows");
    row_mean_f32_scalar<<<dim3(static_cast<unsigned>(blocks)), dim3(256), 0,
                          stream>>>(x, out, rows, cols, row_stride);
  }
  return check_launch("row_mean_f32");
}

extern "C" int hipo_row_mean_bf16(const uint16_t* x, uint16_t* out, int64_t rows,
                                  int64_t cols, int relu, hipStream_t stream) {
  using namespace hipo;
  clear_error();
  HIPO_REQUIRE(rows >= 0 && cols >= 0, "row_mean_bf16: negative size");
  if (rows == 0) return 0;
  HIPO_REQUIRE(cols > 0, "row_mean_bf16: mean over zero elements");
  HIPO_REQUIRE(x != nullptr && out != nullptr, "row_mean_bf16: null pointer");
  const bool act = relu != 0;
  const bool aligned = aligned16(x);
  const bool ragged = cols % 8 != 0 || !aligned;
  const auto blocks_of = [&](int64_t rows_per_block) {
    return (rows + rows_per_block - 1) / rows_per_block;
  };
  // Rows of up to 512 values off 16-byte alignment, us, a wave per row by single
  // values / the short-row kernel / the rows kernel with one load: [10000, 100]
  // 3.3 / 3.9 / 4.2, [100000, 100] 15.6 / 10.3 / 20.0, [100000, 256] 23.8 / 16.2
  // / 20.3, [10000, 400] 6.5 / 7.9 / 4.8, [100000, 400] 35.1 / 23.7 / 20.2; the
  // short-row kernel passes the first at about 24000 rows.
  const bool off_short = !aligned && cols >= kRowGroup && cols <= 256;
  // Whole longer rows: the rows kernel holds `held` values a row, in one sweep
  // of 2 loads a lane or several of 4.
  const int waves = static_cast<int>(
      std::min<int64_t>(kMaxWaves, (cols + 2 * kRowSweep - 1) / (2 * kRowSweep)));
  const bool two = cols <= int64_t{waves} * 2 * kRowSweep;
  const int64_t sweep = int64_t{waves} * (two ? 2 : 4) * kRowSweep;
  const int64_t held = (cols + sweep - 1) / sweep * sweep;
  const int64_t fill = cols * 100 / held;
  // A wave per row is faster where many rows fill little of that, and where
  // one or two waves a row come to more workgroups than CUs.  The rows kernel's
  // time over the wave's, graph replays, 700 points of 520 to 12296 values and 1
  // to 60000 rows.  One wave: 520 values, 2048 rows 1.02, 2300 1.17, 60000 1.08;
  // 704, 24000 rows 1.04 (1.08 with ReLU), 32000 1.01 (1.07), 50000 0.95; 776,
  // 3600 rows 1.16, 16000 1.07, 32000 0.95; 1024, 2300 rows 1.14, 24000 0.99.
  // Two: 1032 values 1.02 to 1.37 from 1400 rows on; 1224, 1400 rows 1.02, 1600
  // 1.13; 1448, 1500 rows 0.93, 2800 1.12; 1736, 3400 rows 1.00, 5000 1.12. Three:
  // 2056 values, 2600 rows 1.01, 3200 1.06; 2312, 2800 rows 0.97, 4000 1.07.
  // More: 4104 values, 3400 rows 0.95, 5000 1.10; 8200, 4096 rows 1.17; 10248,
  // 5000 rows 1.07, 12296, 4096 rows 0.93.
  const int64_t wave_from = waves == 1   ? 2049
                            : waves == 2 ? (fill < 54 ? 1 : fill < 76 ? 1537 : 4096)
                            : waves <= 4 ? (fill < 70 ? 2816 : 3584)
                                         : 4096;
  const bool little = waves == 1 ? fill < 60 || rows <= (fill < 70 ? 32768 : 16384)
                                 : fill < (two ? 85 : 60);
  const bool wave_rows = !ragged && little && rows >= wave_from;
  if (cols <= kBf16ShortCols && (aligned || (off_short && rows >= kBf16ShortRows))) {
    const int64_t blocks = blocks_of(kBf16Waves * kBf16RowsPerWave);
    HIPO_REQUIRE(blocks <= 0x7fffffff, "row_mean_bf16: too many rows");
    // cols vectors of 16 bytes per wave: ceil(cols / 64) per lane.
#define HIPO_RMB(V_)                                                                          \
  (act ? (aligned ? row_mean_bf16_short<true, V_, true> : row_mean_bf16_short<true, V_, false>) \
       : (aligned ? row_mean_bf16_short<false, V_, true> : row_mean_bf16_short<false, V_, false>))
    auto kernel = cols <= 2 * kWave ? HIPO_RMB(2) : cols <= 4 * kWave ? HIPO_RMB(4) : HIPO_RMB(8);
#undef HIPO_RMB
    kernel<<<dim3(static_cast<unsigned>(blocks)), dim3(kBf16Waves * kWave), 0, stream>>>(
        x, out, rows, static_cast<int>(cols));
  } else if (cols < kRowGroup) {
    const int64_t blocks = blocks_of(256);
    HIPO_REQUIRE(blocks <= 0x7fffffff, "row_mean_bf16: too many rows");
    auto kernel = act ? row_mean_bf16_scalar<true> : row_mean_bf16_scalar<false>;
    kernel<<<dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream>>>(x, out, rows, cols);
  } else if (off_short || wave_rows) {
    const int64_t blocks = blocks_of(kBf16Waves);
    HIPO_REQUIRE(blocks <= 0x7fffffff, "row_mean_bf16: too many rows");
#define HIPO_RMB(VEC_) (act ? row_mean_bf16_wave<true, VEC_> : row_mean_bf16_wave<false, VEC_>)
    auto kernel = wave_rows ? HIPO_RMB(true) : HIPO_RMB(false);
#undef HIPO_RMB
    kernel<<<dim3(static_cast<unsigned>(blocks)), dim3(kBf16Waves * kWave), 0, stream>>>(
        x, out, rows, cols);
  } else {
    // Workgroups of 4 waves where 2 to 4 of them make a row (8 / 4 waves, us:
    // [1500, 1448] 3.18 / 2.93, [1280, 1640] 3.05 / 2.73, [9000, 3592] 11.3 / 10.7,
    // [16000, 2312] 14.6 / 13.2), 8 for rows of one wave and two loads (even) and
    // for many ragged rows of 3 and 4 waves (2880 to 4095 values, 1500 rows 0.98,
    // 5000 to 16000 rows 1.05 times the 8 waves' time).
    const bool one = cols <= kRowSweep;
    const bool small_groups =
        one || waves == 2 || (waves > 2 && waves <= kBf16Waves && (!ragged || rows <= 2048));
    const int rpb = (small_groups ? kBf16Waves : kMaxWaves) / waves;
    const int64_t blocks = blocks_of(rpb);
    HIPO_REQUIRE(blocks <= 0x7fffffff, "row_mean_bf16: too many rows");
#define HIPO_RMB(ACT_)                                                                     \
  (one   ? row_mean_bf16_rows<ACT_, 1, true>                                               \
   : two ? (ragged ? row_mean_bf16_rows<ACT_, 2, true> : row_mean_bf16_rows<ACT_, 2, false>) \
         : (ragged ? row_mean_bf16_rows<ACT_, 4, true> : row_mean_bf16_rows<ACT_, 4, false>))
    auto kernel = act ? HIPO_RMB(true) : HIPO_RMB(false);
#undef HIPO_RMB
    kernel<<<dim3(static_cast<unsigned>(blocks)), dim3(waves * rpb * kWave), 0, stream>>>(
        x, out, rows, cols, waves, rpb);
  }
  return check_launch("row_mean_bf16");
}
