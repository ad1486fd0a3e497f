// BatchNorm training forward, fp32 NCHW: per-channel statistics over
// (N, H, W), normalisation + affine (+ ReLU), running-stat update.
//
// Entry point.  Channels of at most 16384 values, and larger ones where that
// measured faster (kLargeChannel), take one launch with a workgroup per
// channel that holds its channel in registers (bn_channel_small).  Other
// channels take the single-pass persistent kernel (batchnorm_fused.hip)
// wherever it applies, and the split-K path below otherwise (HW not a
// multiple of 4, unaligned pointers, very large tensors, more than 64
// workgroups per channel or 64 rounds).
//
// Split-K structure (two launches on the caller's stream):
//   1. bn_partial_stats: S x C workgroups.  Workgroup (s, c) reduces the planes
//      n in [s*N/S, (s+1)*N/S) of channel c to a Welford triple
//      (count, mean, M2) and writes it to the workspace.  Inside the
//      workgroup each thread reduces its slice of every plane exactly
//      (two-pass over registers) and merges it into a running triple with
//      Chan's formula; threads then merge across the wave with DPP and
//      across waves through LDS.
//   2. bn_normalize: S x C workgroups.  The first wave of each merges the S
//      triples of its channel (fp64, fixed order), derives
//      mean / invstd, and writes y = relu?(x * alpha + beta') for its planes
//      with alpha = invstd * gamma, beta' = beta - mean * alpha.  Workgroup
//      (0, c) also writes save_mean / save_invstd and updates the running
//      statistics (unbiased variance, count / (count - 1)).
// This path reads x twice (once per launch).
#include <mutex>
#include <type_traits>

#include "welford.h"

namespace hipo {
namespace {

constexpr int kThreads = 256;

// max(v, 0) that keeps NaN (torch.relu propagates NaN; fmaxf would not).
__device__ __forceinline__ float relu_f32(float v) { return v < 0.f ? 0.f : v; }

// Exact statistics of up to 4*U values held by one thread, merged into acc.
template <int U>
__device__ __forceinline__ void absorb(Welford& acc, const float4 (&v)[U],
                                       const bool (&ok)[U]) {
  float cnt = 0.f, s = 0.f;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (ok[u]) {
      cnt += 4.f;
      s += (v[u].x + v[u].y) + (v[u].z + v[u].w);
    }
  }
  if (cnt == 0.f) return;
  const float m = s / cnt;
  float q = 0.f;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (ok[u]) {
      const float a = v[u].x - m, b = v[u].y - m, c = v[u].z - m, d = v[u].w - m;
      q += (a * a + b * b) + (c * c + d * d);
    }
  }
  acc = welford_merge(acc, Welford{cnt, m, q});
}

// The same for up to U vectors whose first skip[u] values (4: all) belong to
// another vector.
template <int U>
__device__ __forceinline__ void absorb(Welford& acc, const f32x4_t (&v)[U],
                                       const int (&skip)[U]) {
  float cnt = 0.f, s = 0.f;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    cnt += static_cast<float>(4 - skip[u]);
#pragma unroll
    for (int e = 0; e < 4; ++e) s += e >= skip[u] ? v[u][e] : 0.f;
  }
  if (cnt == 0.f) return;
  const float m = s / cnt;
  float q = 0.f;
#pragma unroll
  for (int u = 0; u < U; ++u) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float d = e >= skip[u] ? v[u][e] - m : 0.f;
      q = __builtin_fmaf(d, d, q);
    }
  }
  acc = welford_merge(acc, Welford{cnt, m, q});
}

// The same for up to U single values.
template <int U>
__device__ __forceinline__ void absorb(Welford& acc, const float (&v)[U], const bool (&ok)[U]) {
  float cnt = 0.f, s = 0.f;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (ok[u]) {
      cnt += 1.f;
      s += v[u];
    }
  }
  if (cnt == 0.f) return;
  const float m = s / cnt;
  float q = 0.f;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (ok[u]) q += (v[u] - m) * (v[u] - m);
  }
  acc = welford_merge(acc, Welford{cnt, m, q});
}

// Planes handled by split s of S over N planes.
__device__ __forceinline__ void split_range(int64_t N, int64_t S, int64_t s,
                                            int64_t& n0, int64_t& n1) {
  n0 = (N * s) / S;
  n1 = (N * (s + 1)) / S;
}

// Merge the threads' triples: DPP across the wave, then the four waves'
// triples, through LDS, by the same butterflies in every wave, of which lane
// 0's order counts.  Every thread returns the workgroup's total.
__device__ __forceinline__ Welford block_welford(Welford acc) {
  constexpr int kWaves = kThreads / kWave;
  static_assert(kWaves == 4, "the waves' triples fill quads");
  acc = wave_welford(acc);
  __shared__ Welford part[kWaves];
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & (kWave - 1)) == 0) part[wave] = acc;
  __syncthreads();
  Welford w = part[threadIdx.x & (kWaves - 1)];
  w = welford_merge(w, welford_dpp<kDppQuadXor1>(w));
  w = welford_merge(w, welford_dpp<kDppQuadXor2>(w));
  return welford_lane(w, 0);
}

// Triples (n_s, mean_s, M2_s) merged in fp64 about a shift K, one of the means
// (shift_of it: 0 where it is not finite, for mean_s - K of an infinite one
// would be NaN): with d_s = mean_s - K, S1 = sum n_s d_s and S2 = sum M2_s +
// n_s d_s^2, mean = K + S1 / N and M2 = S2 - S1^2 / N.  Each lane add()s its
// triples in order; total() adds the lanes by wave_sum (a fixed order; all 64
// lanes active, every lane gets the result).
struct ChannelStats {
  double mean, m2, count;
};

__device__ __forceinline__ double shift_of(float mean) {
  return __builtin_isfinite(mean) ? static_cast<double>(mean) : 0.0;
}

struct ShiftedSums {
  double K, n, s1, s2;
  __device__ __forceinline__ void add(float nb, float mean, float m2) {
    const double d = static_cast<double>(mean) - K;
    n += nb;
    s1 = __builtin_fma(static_cast<double>(nb), d, s1);
    s2 += __builtin_fma(nb * d, d, static_cast<double>(m2));
  }
  __device__ __forceinline__ ChannelStats total() const {
    const double N = wave_sum(n), a = wave_sum(s1), b = wave_sum(s2);
    const double dm = a / N;
    // max (NaN from the data kept): rounding can leave a tiny negative.
    return ChannelStats{K + dm, __builtin_elementwise_maximum(b - a * dm, 0.0), N};
  }
};

// Planes of HW >= 4 values, any alignment, as F = ceil(HW / 4) vectors each:
// vector j of a plane starts at value min(4 j, HW - 4), so the last one of a
// plane that is not a whole number of vectors ends with it, and its first
// 4 j - start values (`skip`) are its neighbour's.  16-byte accesses at value
// alignment; a value that two vectors share is normalised by both to the
// same bits.
struct PlaneGeom {
  int64_t HW;
  int F;  // 1 for planes of 2^30 values and more, which go value by value
  DivMagic by_F;
};

inline PlaneGeom plane_geom(int64_t hw) {
  PlaneGeom g;
  g.HW = hw;
  g.F = hw < (int64_t{1} << 30) ? static_cast<int>((hw + 3) / 4) : 1;
  g.by_F = div_magic(static_cast<uint32_t>(g.F));
  return g;
}

struct PlaneVec {
  int64_t off;  // value offset, planes `stride` values apart
  int skip;
};

__device__ __forceinline__ PlaneVec plane_vec(const PlaneGeom& g, int64_t stride, uint32_t i) {
  const uint32_t n = div_by(i, g.by_F);
  const int first = static_cast<int>(i - n * static_cast<uint32_t>(g.F)) * 4;
  const int last = static_cast<int>(g.HW) - 4;
  const int start = first < last ? first : last;
  return PlaneVec{static_cast<int64_t>(n) * stride + start, first - start};
}

constexpr int kSplitLoads = 8;  // vectors in flight per thread

// Welford triple of planes [n0, n1) of channel c over the workgroup: each
// thread reduces its values exactly (two-pass over registers), kSplitLoads
// vectors of consecutive planes at a time, and merges them into a running
// triple with Chan's formula; the wave merges with DPP and the waves through
// LDS.  Thread 0 returns the total.
template <bool VEC>
__device__ Welford planes_welford(const float* __restrict__ x, int64_t n0, int64_t n1,
                                  int64_t C, const PlaneGeom& g, int64_t c) {
  Welford acc{0.f, 0.f, 0.f};
  const int64_t HW = g.HW;
  if constexpr (VEC) {
    const float* base = x + (n0 * C + c) * HW;
    const uint32_t total = static_cast<uint32_t>(n1 - n0) * static_cast<uint32_t>(g.F);
    for (uint32_t i0 = threadIdx.x; i0 < total; i0 += kThreads * kSplitLoads) {
      f32x4_t v[kSplitLoads];
      int skip[kSplitLoads];
#pragma unroll
      for (int u = 0; u < kSplitLoads; ++u) {
        const uint32_t i = i0 + static_cast<uint32_t>(u) * kThreads;
        const PlaneVec p = plane_vec(g, C * HW, i < total ? i : i0);
        v[u] = *reinterpret_cast<const f32x4_a4_t*>(base + p.off);
        skip[u] = i < total ? p.skip : 4;
      }
      absorb<kSplitLoads>(acc, v, skip);
    }
  } else {
    for (int64_t n = n0; n < n1; ++n) {
      const float* plane = x + (n * C + c) * HW;
      for (int64_t i = threadIdx.x; i < HW; i += kThreads) {
        acc = welford_merge(acc, Welford{1.f, plane[i], 0.f});
      }
    }
  }
  return block_welford(acc);
}

template <bool VEC>
__global__ __launch_bounds__(kThreads) void bn_partial_stats(
    const float* __restrict__ x, float* __restrict__ ws, int64_t N, int64_t C,
    PlaneGeom g, int64_t S, DivMagic by_S) {
  const uint32_t bid = xcd_order(blockIdx.x, gridDim.x);
  const int64_t c = div_by(bid, by_S);
  const int64_t s = bid - c * S;
  int64_t n0, n1;
  split_range(N, S, s, n0, n1);
  const Welford t = planes_welford<VEC>(x, n0, n1, C, g, c);
  if (threadIdx.x == 0) {
    float* dst = ws + (c * S + s) * 3;
    dst[0] = t.n;
    dst[1] = t.mean;
    dst[2] = t.m2;
  }
}

// The S partial triples of channel c merged about the first one's mean, lane
// l adding splits l, l + 64, ... .
__device__ ChannelStats channel_stats(const float* __restrict__ ws, int64_t c, int64_t S) {
  const float* p = ws + c * S * 3;
  ShiftedSums sums{shift_of(p[1]), 0.0, 0.0, 0.0};
  for (int64_t s = threadIdx.x & (kWave - 1); s < S; s += kWave)
    sums.add(p[3 * s], p[3 * s + 1], p[3 * s + 2]);
  return sums.total();
}

// mean / invstd from the merged (mean, M2, count) of channel c -> the
// affine coefficients (alpha = invstd * gamma, shift = beta - mean * alpha)
// in coef[0..1]; with write_stats, save_mean / save_invstd and the running
// statistics (unbiased variance, count / (count - 1)).
// channel_coefs with gamma[c], beta[c] and the running statistics already
// loaded (g, b, rm, rv).
__device__ void channel_coefs_of(double mean, double m2, double count, int64_t c, float g,
                                 float b, float rm, float rv, float* __restrict__ running_mean,
                                 float* __restrict__ running_var, float* __restrict__ save_mean,
                                 float* __restrict__ save_invstd, float momentum, float eps,
                                 bool write_stats, float* coef) {
  const float meanf = static_cast<float>(mean);
  const float var = static_cast<float>(m2 / count);
  const float invstd = 1.0f / __builtin_sqrtf(var + eps);
  const float alpha = invstd * g;
  coef[0] = alpha;
  coef[1] = b - meanf * alpha;
  if (write_stats) {
    save_mean[c] = meanf;
    save_invstd[c] = invstd;
    const double unbiased = count > 1.0 ? m2 / (count - 1.0) : __builtin_nan("");
    const double mom = momentum;
    running_mean[c] = static_cast<float>(mom * mean + (1.0 - mom) * rm);
    running_var[c] = static_cast<float>(mom * unbiased + (1.0 - mom) * rv);
  }
}

__device__ void channel_coefs(double mean, double m2, double count, int64_t c,
                              const float* __restrict__ gamma, const float* __restrict__ beta,
                              float* __restrict__ running_mean, float* __restrict__ running_var,
                              float* __restrict__ save_mean, float* __restrict__ save_invstd,
                              float momentum, float eps, bool write_stats, float* coef) {
  channel_coefs_of(mean, m2, count, c, gamma[c], beta[c], write_stats ? running_mean[c] : 0.f,
                   write_stats ? running_var[c] : 0.f, running_mean, running_var, save_mean,
                   save_invstd, momentum, eps, write_stats, coef);
}

// y = relu?(x * alpha + shift) over planes [n0, n1) of channel c.
template <bool VEC>
__device__ void normalize_planes(const float* __restrict__ x, float* __restrict__ y,
                                 int64_t n0, int64_t n1, int64_t C, const PlaneGeom& g,
                                 int64_t c, float alpha, float shift, int relu) {
  const int64_t HW = g.HW;
  if constexpr (VEC) {
    const int64_t base = (n0 * C + c) * HW;
    const uint32_t total = static_cast<uint32_t>(n1 - n0) * static_cast<uint32_t>(g.F);
    for (uint32_t i0 = threadIdx.x; i0 < total; i0 += kThreads * kSplitLoads) {
      f32x4_t v[kSplitLoads];
      int64_t off[kSplitLoads];
#pragma unroll
      for (int u = 0; u < kSplitLoads; ++u) {
        const uint32_t i = i0 + static_cast<uint32_t>(u) * kThreads;
        off[u] = plane_vec(g, C * HW, i < total ? i : i0).off;
        v[u] = *reinterpret_cast<const f32x4_a4_t*>(x + base + off[u]);
      }
#pragma unroll
      for (int u = 0; u < kSplitLoads; ++u) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[u][e] = __builtin_fmaf(v[u][e], alpha, shift);
          if (relu) v[u][e] = relu_f32(v[u][e]);
        }
        if (i0 + static_cast<uint32_t>(u) * kThreads < total)
          *reinterpret_cast<f32x4_a4_t*>(y + base + off[u]) = v[u];
      }
    }
  } else {
    for (int64_t n = n0; n < n1; ++n) {
      const int64_t off = (n * C + c) * HW;
      for (int64_t i = threadIdx.x; i < HW; i += kThreads) {
        float v = __builtin_fmaf(x[off + i], alpha, shift);
        if (relu) v = relu_f32(v);
        y[off + i] = v;
      }
    }
  }
}

template <bool VEC>
__global__ __launch_bounds__(kThreads) void bn_normalize(
    const float* __restrict__ x, const float* __restrict__ gamma,
    const float* __restrict__ beta, float* __restrict__ running_mean,
    float* __restrict__ running_var, float* __restrict__ y,
    float* __restrict__ save_mean, float* __restrict__ save_invstd,
    const float* __restrict__ ws, int64_t N, int64_t C, PlaneGeom g, int64_t S, DivMagic by_S,
    float momentum, float eps, int relu) {
  const uint32_t bid = xcd_order(blockIdx.x, gridDim.x);
  const int64_t c = div_by(bid, by_S);
  const int64_t s = bid - c * S;
  __shared__ float coef[2];
  if (threadIdx.x < kWave) {
    const ChannelStats t = channel_stats(ws, c, S);
    if (threadIdx.x == 0)
      channel_coefs(t.mean, t.m2, t.count, c, gamma, beta, running_mean, running_var, save_mean,
                    save_invstd, momentum, eps, s == 0, coef);
  }
  __syncthreads();
  int64_t n0, n1;
  split_range(N, S, s, n0, n1);
  normalize_planes<VEC>(x, y, n0, n1, C, g, c, coef[0], coef[1], relu);
}

// Small channels (N * HW <= kSmallChannel values): one launch, a workgroup
// per channel holding the channel in registers -- U float4 (or U single
// values when HW % 4 != 0 or x, y are unaligned) per thread, every load in
// flight at once, with gamma, beta and the running statistics loaded beside
// them.  Exact per-thread statistics (two-pass over the registers), Chan
// merges across the wave and the workgroup, fp64 coefficients (the split-K
// path's arithmetic with one split), then y written from the registers: x
// is read once, and the chain from launch to the last store holds a single
// memory round trip for the data.  At ragged points such as [3, 5, 7, 7]
// or [4, 24, 10, 10] that chain, not the bytes, is the time (the
// single-pass kernel adds an epoch read and a slab exchange to it).
constexpr int64_t kSmallChannel = 16384;
// Larger ones take the same kernel with 1024 threads: whole float4 planes up
// to 7 a thread (28672 values; two workgroups per CU) and at least 32
// channels, ragged ones, whose alternative reads x twice, up to 8 vectors a
// thread, and up to 12 in planes below 1024 values or 32 channels and more.
// Graph replays in us, single-pass kernel / here, inputs reused [not reused]: [128, 1024, 14, 14] 56.7 / 39.3 [57.3 / 47.7], [128, 256, 14, 14]
// 15.6 / 11.9 [16.5 / 14.8], [128, 64, 14, 14] 9.2 / 7.1 [9.6 / 8.6], but
// [64, 512, 28, 28], 50176 values, 37.7 / 40.5 [37.8 / 52.0] and [6, 960, 72,
// 70], 30240, 52.4 / 47.8 [52.8 / 57.8].  Split-K before / split-K now / here:
// [512, 512, 7, 7] 95 / 34.5 / 23.0, [17, 488, 35, 37] 41.2 / 32.5 / 19.4, [21,
// 782, 46, 43] 119 / 81 / 58, [12, 1280, 46, 45] 105 / 78 / 53; with 16 vectors
// a thread (and spills) [5, 32, 101, 99] 22.7 / 9.7 / 12.3.  Ragged planes of
// few channels, split-K / here: up to 8 vectors a thread here is faster down to
// one channel ([2, 1, 99, 101] 8.9 / 6.7, [400, 4, 7, 7] 11.6 / 7.0); beyond, only
// for planes that are short ([900, 1, 7, 7] 11.5 / 9.7, but [16, 1, 47, 47] 7.5 /
// 9.1, [16, 16, 47, 47] 7.9 / 9.6, [3, 4, 127, 127] 10.1 / 10.2; from 32 channels
// on they are even).
constexpr int64_t kLargeChannel = 65536;
constexpr int kLargeThreads = 1024;
constexpr int64_t kLargeMinChannels = 32;

// Planes that are not whole float4s, or not 16-byte aligned, are cut into
// vectors at value alignment (PlaneGeom); planes below 9 values that are not
// a multiple of 4, where over a third of those vectors' values would be
// read twice, go value by value.  Workgroups in XCD order: neighbouring
// channels share the cache lines at their planes' ends.  [128, 2048, 7, 7]
// 39.0 us value by value -> 19.0 (5.4 TB/s).  Whole planes of 4 KiB and more,
// which share few, in launch order: [1, 300, 16000] 10.8 us against 11.5, [1,
// 600, 10708] 11.5 against 12.0, [4, 600, 2676] 11.5 against 11.9; but [64, 512,
// 196] 11.6 against 11.4.
struct SmallGeom {
  int total;      // vectors, or values, per channel
  int per_plane;  // HW / 4 (kWhole) or HW (kValues)
  DivMagic by_plane;
  PlaneGeom ragged;  // kRagged
  bool xcd;          // kWhole: workgroups in XCD order (the others always)
};

enum class SmallKind { kValues, kWhole, kRagged };

template <SmallKind KIND, int U, int T>
__global__ __launch_bounds__(T) void bn_channel_small(
    const float* __restrict__ x, const float* __restrict__ gamma,
    const float* __restrict__ beta, float* __restrict__ running_mean,
    float* __restrict__ running_var, float* __restrict__ y,
    float* __restrict__ save_mean, float* __restrict__ save_invstd, SmallGeom g, int64_t C,
    float momentum, float eps, int relu) {
  constexpr bool kVec = KIND != SmallKind::kValues;
  constexpr bool kRagged = KIND == SmallKind::kRagged;
  using Elem = std::conditional_t<kRagged, f32x4_t, std::conditional_t<kVec, float4, float>>;
  const bool xcd = KIND != SmallKind::kWhole || g.xcd;
  const int64_t c = xcd ? xcd_order(blockIdx.x, gridDim.x) : blockIdx.x;
  float pg = 0.f, pb = 0.f, prm = 0.f, prv = 0.f;
  if (threadIdx.x == 0) {
    pg = gamma[c];
    pb = beta[c];
    prm = running_mean[c];
    prv = running_var[c];
  }
  // Element i of the channel: plane i / per_plane, offset i % per_plane
  // (in units of Elem; kRagged: the vector's value offset and its skip).
  auto offset = [&](int i) {
    if constexpr (kRagged) {
      PlaneVec p = plane_vec(g.ragged, C * g.ragged.HW, static_cast<uint32_t>(i));
      p.off += c * g.ragged.HW;
      return p;
    } else {
      const uint32_t n = div_by(static_cast<uint32_t>(i), g.by_plane);
      return (static_cast<int64_t>(n) * C + c) * g.per_plane +
             (i - static_cast<int>(n) * g.per_plane);
    }
  };
  Elem v[U];
  bool ok[U];
  int skip[U];
  // Unconditional loads (threads past the channel's end re-read its last
  // element and store nothing), so all of them are in flight together.
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int i = static_cast<int>(threadIdx.x) + u * T;
    ok[u] = i < g.total;
    const auto at = offset(ok[u] ? i : g.total - 1);
    if constexpr (kRagged) {
      v[u] = *reinterpret_cast<const f32x4_a4_t*>(x + at.off);
      skip[u] = ok[u] ? at.skip : 4;
    } else {
      v[u] = reinterpret_cast<const Elem*>(x)[at];
    }
  }
  Welford acc{0.f, 0.f, 0.f};
  if constexpr (kRagged) {
    absorb<U>(acc, v, skip);
  } else {
    absorb<U>(acc, v, ok);
  }
  __shared__ float coef[2];
  ChannelStats t;
  if constexpr (T == kThreads) {
    const Welford w = block_welford(acc);
    t = ChannelStats{static_cast<double>(w.mean), static_cast<double>(w.m2),
                     static_cast<double>(w.n)};
  } else {
    // The 16 waves' triples in fp64 by the first wave, as the split-K path
    // merges its splits (fp32 merges left the mean up to an ulp and a half
    // off, and the running statistics with it).
    constexpr int kWaves = T / kWave;
    __shared__ Welford part[kWaves];
    acc = wave_welford(acc);
    if ((threadIdx.x & (kWave - 1)) == 0) part[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x < kWave) {
      ShiftedSums sums{shift_of(part[0].mean), 0.0, 0.0, 0.0};
      if (threadIdx.x < kWaves) {
        const Welford w = part[threadIdx.x];
        sums.add(w.n, w.mean, w.m2);
      }
      t = sums.total();
    }
  }
  if (threadIdx.x == 0)
    channel_coefs_of(t.mean, t.m2, t.count, c, pg, pb, prm, prv, running_mean, running_var,
                     save_mean, save_invstd, momentum, eps, true, coef);
  __syncthreads();
  const float alpha = coef[0], shift = coef[1];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (!ok[u]) continue;
    Elem o = v[u];
    if constexpr (kVec) {
      o.x = __builtin_fmaf(o.x, alpha, shift);
      o.y = __builtin_fmaf(o.y, alpha, shift);
      o.z = __builtin_fmaf(o.z, alpha, shift);
      o.w = __builtin_fmaf(o.w, alpha, shift);
      if (relu) {
        o.x = relu_f32(o.x);
        o.y = relu_f32(o.y);
        o.z = relu_f32(o.z);
        o.w = relu_f32(o.w);
      }
    } else {
      o = __builtin_fmaf(o, alpha, shift);
      if (relu) o = relu_f32(o);
    }
    const auto at = offset(static_cast<int>(threadIdx.x) + u * T);
    if constexpr (kRagged) {
      *reinterpret_cast<f32x4_a4_t*>(y + at.off) = o;
    } else {
      reinterpret_cast<Elem*>(y)[at] = o;
    }
  }
}

template <SmallKind KIND, int U, int T = kThreads>
void launch_small(const float* x, const float* gamma, const float* beta, float* running_mean,
                  float* running_var, float* y, float* save_mean, float* save_invstd,
                  const SmallGeom& g, int64_t c, float momentum, float eps, int relu,
                  hipStream_t stream) {
  bn_channel_small<KIND, U, T><<<dim3(static_cast<unsigned>(c)), dim3(T), 0, stream>>>(
      x, gamma, beta, running_mean, running_var, y, save_mean, save_invstd, g, c, momentum,
      eps, relu);
}

// Launches the register-held kernel, U = the smallest instantiated count
// covering the channel; -1 if it does not take the shape.
int small_launch(const float* x, const float* gamma, const float* beta, float* running_mean,
                 float* running_var, float* y, float* save_mean, float* save_invstd, int64_t n,
                 int64_t c, int64_t hw, float momentum, float eps, int relu,
                 hipStream_t stream) {
  if (c > 0x7fffffff || hw > kLargeChannel || n * hw > kLargeChannel) return -1;
  const bool whole = hw % 4 == 0 && aligned16(x) && aligned16(y);
  const bool ragged = !whole && (hw % 4 == 0 || hw >= 9);
  SmallGeom g;
  g.per_plane = static_cast<int>(whole ? hw / 4 : hw);
  g.by_plane = div_magic(static_cast<uint32_t>(g.per_plane));
  g.ragged = plane_geom(hw);
  g.xcd = hw < 1024;
  g.total = static_cast<int>(n) * (ragged ? g.ragged.F : g.per_plane);
#define HIPO_BN_SMALL(K, ...)                                                        \
  launch_small<SmallKind::K, __VA_ARGS__>(x, gamma, beta, running_mean, running_var, y, \
                                          save_mean, save_invstd, g, c, momentum, eps,  \
                                          relu, stream)
  if (n * hw > kSmallChannel) {
    const int per_thread = (g.total + kLargeThreads - 1) / kLargeThreads;
    if (whole && c >= kLargeMinChannels && per_thread <= 7)
      HIPO_BN_SMALL(kWhole, 7, kLargeThreads);
    else if (ragged && per_thread <= 8)
      HIPO_BN_SMALL(kRagged, 8, kLargeThreads);
    else if (ragged && per_thread <= 12 && (c >= kLargeMinChannels || hw < 1024))
      HIPO_BN_SMALL(kRagged, 12, kLargeThreads);
    else
      return -1;
    return check_launch("batchnorm_train_fwd_f32 (channels in registers)");
  }
  const int per_thread = (g.total + kThreads - 1) / kThreads;
  if (whole) {
    if (per_thread <= 1) HIPO_BN_SMALL(kWhole, 1);
    else if (per_thread <= 2) HIPO_BN_SMALL(kWhole, 2);
    else if (per_thread <= 4) HIPO_BN_SMALL(kWhole, 4);
    else if (per_thread <= 8) HIPO_BN_SMALL(kWhole, 8);
    else HIPO_BN_SMALL(kWhole, 16);
  } else if (ragged) {
    // At most 16384 values in planes of 9 or more: 12 / 9 of them in
    // vectors, 21.3 a thread.
    if (per_thread <= 1) HIPO_BN_SMALL(kRagged, 1);
    else if (per_thread <= 2) HIPO_BN_SMALL(kRagged, 2);
    else if (per_thread <= 4) HIPO_BN_SMALL(kRagged, 4);
    else if (per_thread <= 8) HIPO_BN_SMALL(kRagged, 8);
    else if (per_thread <= 16) HIPO_BN_SMALL(kRagged, 16);
    else HIPO_BN_SMALL(kRagged, 24);
  } else {
    if (per_thread <= 1) HIPO_BN_SMALL(kValues, 1);
    else if (per_thread <= 4) HIPO_BN_SMALL(kValues, 4);
    else if (per_thread <= 16) HIPO_BN_SMALL(kValues, 16);
    else HIPO_BN_SMALL(kValues, 64);
  }
#undef HIPO_BN_SMALL
  return check_launch("batchnorm_train_fwd_f32 (small channels)");
}

// Number of plane splits per channel for the split-K launches.
int64_t num_splits(int64_t n, int64_t c) {
  const int64_t target_blocks = 4096;
  int64_t s = (target_blocks + c - 1) / c;
  if (s > n) s = n;
  if (s < 1) s = 1;
  return s;
}

}  // namespace
}  // namespace hipo

extern "C" size_t hipo_batchnorm_workspace_bytes(int64_t n, int64_t c,
                                                 int64_t hw) {
  if (n <= 0 || c <= 0 || hw <= 0) return 0;
  const int64_t s = hipo::num_splits(n, c);
  return hipo::kBnCtlBytes + hipo::bn_fused_slot_bytes(n, c, hw) +
         static_cast<size_t>(c * s * 3) * sizeof(float);
}

extern "C" int hipo_batchnorm_train_fwd_f32(
    const float* x, const float* gamma, const float* beta, float* running_mean,
    float* running_var, float* y, float* save_mean, float* save_invstd,
    int64_t n, int64_t c, int64_t hw, float momentum, float eps, int relu,
    void* workspace, size_t workspace_bytes, hipStream_t stream) {
  using namespace hipo;
  clear_error();
  HIPO_REQUIRE(n > 0 && c > 0 && hw > 0, "batchnorm: sizes must be positive");
  HIPO_REQUIRE(x && gamma && beta && running_mean && running_var && y &&
                   save_mean && save_invstd && workspace,
               "batchnorm: null pointer");
  const size_t need = hipo_batchnorm_workspace_bytes(n, c, hw);
  HIPO_REQUIRE(workspace_bytes >= need,
               "batchnorm: workspace %zu bytes < required %zu", workspace_bytes,
               need);
  HIPO_REQUIRE(reinterpret_cast<uintptr_t>(workspace) % 8 == 0,
               "batchnorm: workspace must be 8-byte aligned");
  const int held = small_launch(x, gamma, beta, running_mean, running_var, y, save_mean,
                                save_invstd, n, c, hw, momentum, eps, relu, stream);
  if (held >= 0) return held;
  const int fused = bn_fused_launch(x, gamma, beta, running_mean, running_var, y,
                                    save_mean, save_invstd, n, c, hw, momentum,
                                    eps, relu, workspace, stream);
  if (fused >= 0) return fused;

  HIPO_REQUIRE(c <= 65535, "batchnorm: too many channels");
  const int64_t S = num_splits(n, c);
  const PlaneGeom g = plane_geom(hw);
  const bool vec = hw >= 4 && hw < (int64_t{1} << 30) &&
                   (n + S - 1) / S * g.F < (int64_t{1} << 30);
  // In place (y == x), planes whose last vector is moved back go value by
  // value in the second pass: the values it shares with its neighbour would
  // be read by one thread after the other stored them.
  const bool apply_vec = vec && (hw % 4 == 0 || y != x);
  const dim3 grid(static_cast<unsigned>(S * c));
  const DivMagic by_S = div_magic(static_cast<uint32_t>(S));
  float* ws = reinterpret_cast<float*>(static_cast<char*>(workspace) + kBnCtlBytes +
                                       bn_fused_slot_bytes(n, c, hw));
  auto stats = vec ? bn_partial_stats<true> : bn_partial_stats<false>;
  stats<<<grid, dim3(kThreads), 0, stream>>>(x, ws, n, c, g, S, by_S);
  int rc = check_launch("batchnorm_train_fwd_f32 (stats)");
  if (rc) return rc;
  auto normalize = apply_vec ? bn_normalize<true> : bn_normalize<false>;
  normalize<<<grid, dim3(kThreads), 0, stream>>>(x, gamma, beta, running_mean, running_var, y,
                                                 save_mean, save_invstd, ws, n, c, g, S, by_S,
                                                 momentum, eps, relu);
  return check_launch("batchnorm_train_fwd_f32 (normalize)");
}

// ---------------------------------------------------------------------------
// Allocation-free variant: the workspace is a file-scope device array.
//
// Each device the library runs on holds its own copy of `scratch`, for the
// life of the process.  On the host the array's name is only a stand-in for
// that memory: its device address is looked up once per device
// (hipGetSymbolAddress, with that device current) and only that address is
// passed to kernels.  The first call on a device also clears the array with
// a fill kernel on the caller's stream and waits for it (that first call
// synchronises; later ones do not): the single-pass kernel's control words
// (completion count, epoch) must start at zero and its exchange slots must
// carry no tag of a future epoch.  hipo_batchnorm_noalloc_error reads (and
// clears) the array's sticky error word, the one fault signal of this path
// besides the NaN outputs.  After that, the epoch protocol keeps the array consistent from one
// call to the next, for any shape that fits; calls that overlap on one
// device (two streams) race on it.
// ---------------------------------------------------------------------------
namespace hipo {
namespace {

constexpr size_t kBnScratchBytes = size_t{4} << 20;  // 4 MiB per device
static __device__ __align__(256) unsigned char scratch[kBnScratchBytes];

constexpr int kScratchDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kScratchDevices] = {};

__global__ __launch_bounds__(256) void bn_scratch_clear(u32x4_t* __restrict__ p,
                                                       uint32_t n16) {
  for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < n16; i += gridDim.x * 256u)
    p[i] = u32x4_t{0u, 0u, 0u, 0u};
}

// The device address of this device's scratch array, set up (and cleared on
// `stream`) by the first call on the device; nullptr after an error.
void* scratch_for_current_device(hipStream_t stream) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kScratchDevices) {
    set_error("batchnorm (no-alloc): no current device");
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] != nullptr) return g_scratch_ptr[dev];
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) {
    (void)hipGetLastError();
    set_error("batchnorm (no-alloc): the first call on a device sets up its scratch "
              "array and must not be captured; call once outside capture first");
    return nullptr;
  }
  void* ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess || ptr == nullptr) {
    (void)hipGetLastError();
    set_error("batchnorm (no-alloc): hipGetSymbolAddress failed: %s", hipGetErrorString(e));
    return nullptr;
  }
  const uint32_t n16 = static_cast<uint32_t>(kBnScratchBytes / 16);
  bn_scratch_clear<<<dim3(256), dim3(256), 0, stream>>>(static_cast<u32x4_t*>(ptr), n16);
  if (check_launch("batchnorm (no-alloc) scratch clear") != 0) return nullptr;
  // The clear completes before the address is published: a first call on
  // another stream that finds the pointer cannot start while the control
  // words are still being zeroed.
  const hipError_t se = hipStreamSynchronize(stream);
  if (se != hipSuccess) {
    (void)hipGetLastError();
    set_error("batchnorm (no-alloc): scratch clear failed: %s", hipGetErrorString(se));
    return nullptr;
  }
  g_scratch_ptr[dev] = ptr;
  return ptr;
}

}  // namespace
}  // namespace hipo

extern "C" int hipo_batchnorm_train_fwd_f32_noalloc(
    const float* x, const float* gamma, const float* beta, float* running_mean,
    float* running_var, float* y, float* save_mean, float* save_invstd,
    int64_t n, int64_t c, int64_t hw, float momentum, float eps, int relu,
    hipStream_t stream) {
  using namespace hipo;
  clear_error();
  HIPO_REQUIRE(n > 0 && c > 0 && hw > 0, "batchnorm: sizes must be positive");
  const size_t need = hipo_batchnorm_workspace_bytes(n, c, hw);
  HIPO_REQUIRE(need <= kBnScratchBytes,
               "batchnorm (no-alloc): this shape needs %zu bytes of workspace, more "
               "than the %zu-byte scratch array; use hipo_batchnorm_train_fwd_f32",
               need, kBnScratchBytes);
  void* ws = scratch_for_current_device(stream);
  if (ws == nullptr) return HIPO_EINVAL;
  return hipo_batchnorm_train_fwd_f32(x, gamma, beta, running_mean, running_var, y,
                                      save_mean, save_invstd, n, c, hw, momentum, eps,
                                      relu, ws, kBnScratchBytes, stream);
}

extern "C" int hipo_batchnorm_noalloc_error(int device, uint32_t* word, int clear) {
  using namespace hipo;
  clear_error();
  HIPO_REQUIRE(word != nullptr, "batchnorm_noalloc_error: null word pointer");
  *word = 0;
  HIPO_REQUIRE(device >= 0 && device < kScratchDevices,
               "batchnorm_noalloc_error: device %d out of range", device);
  void* ptr = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    ptr = g_scratch_ptr[device];
  }
  if (ptr == nullptr) return 0;  // the entry point never ran on this device
  int cur = -1;
  if (hipGetDevice(&cur) != hipSuccess) cur = -1;
  hipError_t e = hipSetDevice(device);
  unsigned char* err = static_cast<unsigned char*>(ptr) + kBnErrorWordOffset;
  // Every kernel that may set the word has finished before it is read.
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e == hipSuccess) e = hipMemcpy(word, err, sizeof(uint32_t), hipMemcpyDeviceToHost);
  if (e == hipSuccess && clear && *word != 0) {
    const uint32_t zero = 0;
    e = hipMemcpy(err, &zero, sizeof(uint32_t), hipMemcpyHostToDevice);
  }
  if (cur >= 0) (void)hipSetDevice(cur);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    set_error("batchnorm_noalloc_error: %s", hipGetErrorString(e));
    return static_cast<int>(e);
  }
  return 0;
}
