// Fused row reductions (sum, max, stable softmax) and RMSNorm on fp32 rows.
//
// Semantics follow the reference's CPU oracles:
//   sum      binary64 accumulation, rounded to float
//            (internal/prometheus/native/reactor_vulkan_fused_reduction.c:1011-1014)
//   max      float comparison `v > m` (same file :1015-1018)
//   softmax  float row max, sum of exp(x - max), out = exp(x - max) / sum (:1019-1028)
//   rmsnorm  inv = 1 / sqrt(sum(x^2)/W + eps), y = x * inv * w, no mean
//            subtraction (reactor_vulkan_gemma4e2b.c:286-319)
//
// MI355X design (the reference's Vulkan path splits a 4096-wide row into
// 1024-element partial workgroups and runs up to 5 dispatches per softmax,
// PrometheusReduction.concept:128-164).  All of it is bound by HBM, so a row is read
// once and kept in registers, and what varies is how many waves share it:
//   * one wave per row of at most 1024 values;
//   * a workgroup of 4 or 16 waves per row of up to 32768 values (one wave per row
//     left much of the chip idle: RMSNorm of 1056 rows of 3840 values 10.6 us,
//     four waves per row 7.9; 512 rows of 8192 values, softmax, 87 -> 10.2);
//   * wider rows over several workgroups of 8192 values each: one
//     launch leaves each part's sum or (maximum, sum), a second one combines a
//     row's parts and, for softmax and RMSNorm, reads the row again (from the
//     caches where it fits) and writes it.  16 rows of 262144 values, softmax:
//     one wave per row 3165 us, now 15.0 (its 33 MB in the caches).
// Loads and stores are 16 bytes per lane whatever the row's alignment (4 bytes is
// enough for them); a width that is not a multiple of 4 ends in single values.
// Cross-lane steps are wave64 shuffles, cross-wave steps go through LDS; sums
// accumulate in binary64 (free on a bandwidth-bound kernel and closest to the oracle).
#include <algorithm>
#include <mutex>

#include "reactor_internal.h"

namespace prom {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));  // 16 bytes at any float

constexpr uint32_t kOpSum = 1, kOpMax = 2, kOpSoftmax = 3, kOpRms = 4;
constexpr float kLog2e = 1.4426950408889634f;

// Hardware base-2 exponential (v_exp_f32).
__device__ __forceinline__ float exp2_hw(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// `v > m` keeps the oracle's rule: a NaN counts only as the starting value.
__device__ __forceinline__ float wave_max_f32(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float o = __shfl_xor(v, off, 64);
    v = o > v ? o : v;
  }
  return v;
}

// Sum / maximum over the kWR waves that share a row; every lane gets it.
template <int kWR>
__device__ __forceinline__ double row_sum(double v, double* part) {
  v = wave_sum_f64(v);
  if constexpr (kWR > 1) {
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    v = part[0];
#pragma unroll
    for (int i = 1; i < kWR; ++i) v += part[i];
  }
  return v;
}

template <int kWR>
__device__ __forceinline__ float row_max(float v, float* part) {
  v = wave_max_f32(v);
  if constexpr (kWR > 1) {
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    v = part[0];
#pragma unroll
    for (int i = 1; i < kWR; ++i) v = part[i] > v ? part[i] : v;
  }
  return v;
}

// kThreads threads hold up to 4 * kThreads * kChunks values of a row: thread t has
// values 4 (c kThreads + t) .. +3 in chunk c.  kTail: the count need not be a
// multiple of 4.
template <int kThreads, int kChunks, bool kTail>
struct RowTile {
  floatx4 v[kChunks];

  static __device__ __forceinline__ uint32_t at(int c, uint32_t t) { return 4u * ((uint32_t)c * kThreads + t); }

  __device__ __forceinline__ void load(const float* __restrict__ src, uint32_t count, uint32_t t) {
#pragma unroll
    for (int c = 0; c < kChunks; ++c) {
      const uint32_t i = at(c, t);
      if (kTail ? i + 4 <= count : i < count) {
        v[c] = *reinterpret_cast<const floatx4u*>(src + i);
      } else if (kTail && i < count) {
#pragma unroll
        for (int j = 0; j < 3; ++j) v[c][j] = i + j < count ? src[i + j] : 0.0f;
      }
    }
  }

  __device__ __forceinline__ void store(float* __restrict__ dst, uint32_t count, uint32_t t) const {
#pragma unroll
    for (int c = 0; c < kChunks; ++c) {
      const uint32_t i = at(c, t);
      if (kTail ? i + 4 <= count : i < count) {
        *reinterpret_cast<floatx4u*>(dst + i) = v[c];
      } else if (kTail && i < count) {
#pragma unroll
        for (int j = 0; j < 3; ++j)
          if (i + j < count) dst[i + j] = v[c][j];
      }
    }
  }

  // f(value, chunk, element) for every value of the row that this thread holds.
  template <class F>
  __device__ __forceinline__ void each(uint32_t count, uint32_t t, F f) {
#pragma unroll
    for (int c = 0; c < kChunks; ++c) {
      const uint32_t i = at(c, t);
      if (i < count) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (!kTail || j == 0 || i + j < count) f(v[c][j], c, j);
      }
    }
  }

  // The same, replacing each value by f's.
  template <class F>
  __device__ __forceinline__ void map(uint32_t count, uint32_t t, F f) {
    each(count, t, [&](float x, int c, int j) { v[c][j] = f(x, c, j); });
  }

  __device__ __forceinline__ double sum(uint32_t count, uint32_t t) {
    double acc = 0.0;
    if constexpr (kTail) {
      each(count, t, [&](float x, int, int) { acc += (double)x; });
    } else {
#pragma unroll
      for (int c = 0; c < kChunks; ++c)
        if (at(c, t) < count) acc += ((double)v[c].x + (double)v[c].y) + ((double)v[c].z + (double)v[c].w);
    }
    return acc;
  }

  __device__ __forceinline__ double sum_squares(uint32_t count, uint32_t t) {
    double acc = 0.0;
    if constexpr (kTail) {
      each(count, t, [&](float x, int, int) { acc += (double)(x * x); });
    } else {
#pragma unroll
      for (int c = 0; c < kChunks; ++c)
        if (at(c, t) < count)
          acc += ((double)(v[c].x * v[c].x) + (double)(v[c].y * v[c].y)) +
                 ((double)(v[c].z * v[c].z) + (double)(v[c].w * v[c].w));
    }
    return acc;
  }

  __device__ __forceinline__ float max(float first, uint32_t count, uint32_t t) {
    float m = first;
    each(count, t, [&](float x, int, int) { m = x > m ? x : m; });
    return m;
  }

  // Replaces the values by exp(v - m).  (v - m) is formed first: it is exact when
  // the two are close, so rows of large nearby values (1e4 +- 8) keep full accuracy.
  // kFast: exp2((v - m) log2 e) on the hardware exp2, a few ulps, for the short
  // aligned rows; the others use expf.
  template <bool kFast>
  __device__ __forceinline__ void exp_minus(float m, uint32_t count, uint32_t t) {
    map(count, t, [&](float x, int, int) { return kFast ? exp2_hw((x - m) * kLog2e) : expf(x - m); });
  }
};

// RMSNorm's scale of a row from its sum of squares.
__device__ __forceinline__ float inv_rms(double sum, uint32_t width, float eps) {
  const float sumsq = (float)sum;
  return 1.0f / sqrtf(sumsq / (float)width + eps);
}

// One row per kWR waves (kWR == 1: four rows per workgroup), width at most
// 256 kWR kChunks.  RMSNorm's weights load with the row: with few rows each wave's
// memory latency is the cost.
template <uint32_t kOp, int kWR, int kChunks, bool kTail>
__global__ __launch_bounds__(kWR == 1 ? 256 : 64 * kWR) void row_kernel(const float* __restrict__ in,
                                                                        const float* __restrict__ w,
                                                                        float* __restrict__ out,
                                                                        float* __restrict__ aux, uint32_t rows,
                                                                        uint32_t width, uint32_t stride, float eps) {
  constexpr int kThreads = 64 * kWR;
  constexpr bool kFast = !kTail && kWR * kChunks <= 16;
  __shared__ double part_d[kWR];
  __shared__ float part_f[kWR];
  const uint32_t t = kWR == 1 ? threadIdx.x & 63 : threadIdx.x;
  const uint32_t row = kWR == 1 ? blockIdx.x * 4u + (threadIdx.x >> 6) : blockIdx.x;
  if (kWR == 1 && row >= rows) return;
  const float* src = in + (size_t)row * stride;
  RowTile<kThreads, kChunks, kTail> x;
  x.load(src, width, t);
  if constexpr (kOp == kOpSum) {
    const double s = row_sum<kWR>(x.sum(width, t), part_d);
    if (t == 0) out[row] = (float)s;
  } else if constexpr (kOp == kOpMax) {
    const float m = row_max<kWR>(x.max(src[0], width, t), part_f);
    if (t == 0) out[row] = m;
  } else if constexpr (kOp == kOpSoftmax) {
    const float m = row_max<kWR>(x.max(src[0], width, t), part_f);
    x.template exp_minus<kFast>(m, width, t);
    const double s = row_sum<kWR>(x.sum(width, t), part_d);
    const float rden = (float)(1.0 / s);  // one correctly rounded reciprocal
    x.map(width, t, [&](float y, int, int) { return y * rden; });
    x.store(out + (size_t)row * width, width, t);
  } else {
    RowTile<kThreads, kChunks, kTail> g;
    g.load(w, width, t);
    const float inv = inv_rms(row_sum<kWR>(x.sum_squares(width, t), part_d), width, eps);
    x.map(width, t, [&](float y, int c, int j) { return y * inv * g.v[c][j]; });
    x.store(out + (size_t)row * width, width, t);
    if (aux != nullptr && t == 0) aux[row] = inv;
  }
}

// Rows over several workgroups: part p of a row is its values [8192 p, 8192 p +
// 8192).  parts[row * n + p] is the part's sum (sum, RMSNorm: of squares), maximum
// (in `max`), or both: (maximum, sum of exp(x - maximum)).
constexpr uint32_t kPartValues = 8192;

struct RowPart {
  double sum;
  float max;
  float pad;
};

template <uint32_t kOp>
__global__ __launch_bounds__(256) void row_parts_kernel(const float* __restrict__ in, RowPart* __restrict__ parts,
                                                        uint32_t n, uint32_t width, uint32_t stride) {
  __shared__ double part_d[4];
  __shared__ float part_f[4];
  const uint32_t row = blockIdx.x / n, p = blockIdx.x - row * n, t = threadIdx.x;
  const float* src = in + (size_t)row * stride;
  const uint32_t count = min(kPartValues, width - p * kPartValues);
  RowTile<256, 8, true> x;
  x.load(src + p * kPartValues, count, t);
  RowPart r{0.0, 0.0f, 0.0f};
  if constexpr (kOp == kOpMax || kOp == kOpSoftmax) r.max = row_max<4>(x.max(src[0], count, t), part_f);
  if constexpr (kOp == kOpSoftmax) {
    // A part of negative infinities alone adds nothing (and NaN where the whole
    // row is that): its sum is finite and gets the factor exp(-inf - maximum).
    x.template exp_minus<false>(r.max == -__builtin_inff() ? 0.0f : r.max, count, t);
  }
  if constexpr (kOp == kOpSum || kOp == kOpSoftmax) r.sum = row_sum<4>(x.sum(count, t), part_d);
  if constexpr (kOp == kOpRms) r.sum = row_sum<4>(x.sum_squares(count, t), part_d);
  if (t == 0) parts[blockIdx.x] = r;
}

// Combines the n parts of a row in every wave, lane l taking parts l, l + 64, ...
template <uint32_t kOp>
__device__ __forceinline__ RowPart combine_parts(const RowPart* __restrict__ parts, uint32_t n) {
  const uint32_t lane = threadIdx.x & 63;
  RowPart r{0.0, parts[0].max, 0.0f};
  if constexpr (kOp == kOpMax || kOp == kOpSoftmax) {
    for (uint32_t i = lane; i < n; i += 64) r.max = parts[i].max > r.max ? parts[i].max : r.max;
    r.max = wave_max_f32(r.max);
  }
  if constexpr (kOp != kOpMax) {
    for (uint32_t i = lane; i < n; i += 64)
      r.sum += kOp == kOpSoftmax ? parts[i].sum * exp((double)parts[i].max - (double)r.max) : parts[i].sum;
    r.sum = wave_sum_f64(r.sum);
  }
  return r;
}

// Sum and max: a wave per row.  Softmax and RMSNorm: a workgroup per part.
template <uint32_t kOp>
__global__ __launch_bounds__(256) void row_finish_kernel(const float* __restrict__ in, const float* __restrict__ w,
                                                         float* __restrict__ out, float* __restrict__ aux,
                                                         const RowPart* __restrict__ parts, uint32_t n, uint32_t rows,
                                                         uint32_t width, uint32_t stride, float eps) {
  if constexpr (kOp == kOpSum || kOp == kOpMax) {
    const uint32_t row = blockIdx.x * 4u + (threadIdx.x >> 6);
    if (row >= rows) return;
    const RowPart r = combine_parts<kOp>(parts + (size_t)row * n, n);
    if ((threadIdx.x & 63) == 0) out[row] = kOp == kOpSum ? (float)r.sum : r.max;
  } else {
    const uint32_t row = blockIdx.x / n, p = blockIdx.x - row * n, t = threadIdx.x;
    const uint32_t count = min(kPartValues, width - p * kPartValues);
    RowTile<256, 8, true> x;
    x.load(in + (size_t)row * stride + p * kPartValues, count, t);
    const RowPart r = combine_parts<kOp>(parts + (size_t)row * n, n);
    if constexpr (kOp == kOpSoftmax) {
      const float rden = (float)(1.0 / r.sum);
      x.template exp_minus<false>(r.max, count, t);
      x.map(count, t, [&](float y, int, int) { return y * rden; });
    } else {
      const float inv = inv_rms(r.sum, width, eps);
      RowTile<256, 8, true> g;
      g.load(w + p * kPartValues, count, t);
      x.map(count, t, [&](float y, int c, int j) { return y * inv * g.v[c][j]; });
      if (aux != nullptr && p == 0 && t == 0) aux[row] = inv;
    }
    x.store(out + (size_t)row * width + p * kPartValues, count, t);
  }
}

// How a call runs: `waves` per row holding `chunks` chunks each, or split rows.
// us at 6 TB/s would be 44.7 for softmax of 8192 rows of 4096: one wave of 16
// chunks 52.1, four of 4 48.6; 4096 rows of 8192: four waves of 8 51.9, sixteen of 4
// 49.4, and sums 23.4 and 24.4 the other way round; 8192 rows of 1000: one wave
// 11.5, four 12.9.  Rows of up to 32768 stay whole while there are enough of them
// (softmax of 1024 rows of 32768: whole 65, split 84; 256 rows: 16.6 and 23.6).
struct RowPlan {
  int waves, chunks;  // waves 0: rows over several workgroups
};

// Split rows' parts are in one buffer: one call queues its launches at a time.  Taken
// after ctx().mu where a caller holds both.
std::mutex g_parts_mu;

size_t parts_bytes(uint32_t width) {
  return ((size_t)width + kPartValues - 1) / kPartValues * sizeof(RowPart);
}

RowPlan plan_rows(uint32_t op, uint32_t rows, uint32_t width) {
  if (width > 32768u || (width > kPartValues && rows <= 32u)) return {0, 0};
  if (width <= 1024u) return {1, width <= 256u ? 1 : 4};
  if (width <= 4096u) return {4, width <= 2048u ? 2 : 4};
  if (width <= 8192u && (op == kOpSum || op == kOpMax)) return {4, 8};
  return {16, width <= 16384u ? 4 : 8};
}

template <uint32_t kOp, bool kTail>
hipError_t launch_rows(RowPlan p, const float* in, const float* w, float* out, float* aux, uint32_t rows,
                       uint32_t width, uint32_t stride, float eps, hipStream_t stream) {
  constexpr bool kScalar = kOp == kOpSum || kOp == kOpMax;
  if (p.waves == 0) {
    const uint32_t n = (uint32_t)(parts_bytes(width) / sizeof(RowPart));
    // The parts' buffer is had with the device; more rows than it holds the parts of go
    // in blocks, one after the other on the stream (2^17 parts are 2^30 values).
    const uint32_t block = std::max(1u, (uint32_t)(kRowPartsBytes / sizeof(RowPart)) / n);
    std::lock_guard<std::mutex> lock(g_parts_mu);
    RowPart* parts = static_cast<RowPart*>(staging(10, std::max(kRowPartsBytes, parts_bytes(width))));
    if (parts == nullptr) return hipErrorOutOfMemory;
    for (uint32_t r = 0; r < rows; r += std::min(block, rows - r)) {
      const uint32_t count = std::min(block, rows - r);
      const float* x = in + (size_t)r * stride;
      hipLaunchKernelGGL((row_parts_kernel<kOp>), dim3(count * n), dim3(256), 0, stream, x, parts, n, width, stride);
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
      const uint32_t blocks = kScalar ? (count + 3u) / 4u : count * n;
      hipLaunchKernelGGL((row_finish_kernel<kOp>), dim3(blocks), dim3(256), 0, stream, x, w,
                         out + (kScalar ? r : (size_t)r * width), aux != nullptr ? aux + r : nullptr, parts, n, count,
                         width, stride, eps);
      const hipError_t e2 = hipGetLastError();
      if (e2 != hipSuccess) return e2;
    }
    return hipSuccess;
  }
  // A launch has fewer than 2^32 threads: more rows go in blocks (RMSNorm of 2^24 rows of
  // four waves each, or 2^22 of sixteen).
  const uint32_t block = (uint32_t)((1ull << 31) / (64u * (uint32_t)p.waves));
#define ROWS(W, C)                                                                                                \
  hipLaunchKernelGGL((row_kernel<kOp, W, C, kTail>), dim3(W == 1 ? (count + 3u) / 4u : count),                    \
                     dim3(W == 1 ? 256 : 64 * W), 0, stream, x, w, y, aux != nullptr ? aux + r : nullptr, count,  \
                     width, stride, eps);                                                                         \
  break
  for (uint32_t r = 0; r < rows; r += std::min(block, rows - r)) {
    const uint32_t count = std::min(block, rows - r);
    const float* x = in + (size_t)r * stride;
    float* y = out + (kScalar ? r : (size_t)r * width);
    switch (p.waves * 100 + p.chunks) {
      case 101: ROWS(1, 1);
      case 104: ROWS(1, 4);
      case 402: ROWS(4, 2);
      case 404: ROWS(4, 4);
      case 408: ROWS(4, 8);
      case 1604: ROWS(16, 4);
      case 1608: ROWS(16, 8);
      default: return hipErrorInvalidValue;
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
#undef ROWS
  return hipSuccess;
}

// Rows of whole 16-byte chunks at 16-byte addresses take the kernels without tails.
template <uint32_t kOp>
hipError_t dispatch(const float* in, const float* w, float* out, float* aux, uint32_t rows, uint32_t width,
                    uint32_t stride, float eps, hipStream_t stream) {
  const RowPlan p = plan_rows(kOp, rows, width);
  const bool whole = width % 4u == 0 && stride == width && (reinterpret_cast<uintptr_t>(in) & 15u) == 0 &&
                     (reinterpret_cast<uintptr_t>(out) & 15u) == 0 && (reinterpret_cast<uintptr_t>(w) & 15u) == 0;
  return whole ? launch_rows<kOp, false>(p, in, w, out, aux, rows, width, stride, eps, stream)
               : launch_rows<kOp, true>(p, in, w, out, aux, rows, width, stride, eps, stream);
}

// The benchmark entry's correctness reference: the same reduction with every
// sum, exponential and quotient in binary64 (one workgroup per row, a
// strided lane pass then an LDS tree), rounded to float at the end.  It shares
// no code with the fp32 kernels above.
__global__ __launch_bounds__(256) void row_reduction_check_kernel(const float* __restrict__ in,
                                                                  float* __restrict__ out, uint32_t width,
                                                                  uint32_t op) {
  __shared__ double part[256];
  const uint32_t lane = threadIdx.x;
  const float* x = in + (size_t)blockIdx.x * width;
  float m = -__builtin_inff();
  if (op != kOpSum) {
    for (uint32_t i = lane; i < width; i += 256) m = x[i] > m ? x[i] : m;
    part[lane] = (double)m;
    __syncthreads();
    for (uint32_t s = 128; s > 0; s >>= 1) {
      if (lane < s && part[lane + s] > part[lane]) part[lane] = part[lane + s];
      __syncthreads();
    }
    m = (float)part[0];
    __syncthreads();
    if (op == kOpMax) {
      if (lane == 0) out[blockIdx.x] = m;
      return;
    }
  }
  double acc = 0.0;
  for (uint32_t i = lane; i < width; i += 256) acc += op == kOpSum ? (double)x[i] : exp((double)x[i] - (double)m);
  part[lane] = acc;
  __syncthreads();
  for (uint32_t s = 128; s > 0; s >>= 1) {
    if (lane < s) part[lane] += part[lane + s];
    __syncthreads();
  }
  const double total = part[0];
  if (op == kOpSum) {
    if (lane == 0) out[blockIdx.x] = (float)total;
    return;
  }
  for (uint32_t i = lane; i < width; i += 256)
    out[(size_t)blockIdx.x * width + i] = (float)(exp((double)x[i] - (double)m) / total);
}

}  // namespace

bool row_parts_allocate(uint32_t width) { return !ctx().row_parts || parts_bytes(width) > kRowPartsBytes; }

hipError_t launch_row_reduction_check(const float* in, float* out, uint32_t rows, uint32_t width, uint32_t op,
                                      hipStream_t stream) {
  if (rows == 0 || width == 0 || op < kOpSum || op > kOpSoftmax) return hipErrorInvalidValue;
  hipLaunchKernelGGL(row_reduction_check_kernel, dim3(rows), dim3(256), 0, stream, in, out, width, op);
  return hipGetLastError();
}

hipError_t launch_row_reduction(const float* in, float* out, uint32_t rows, uint32_t width, uint32_t op,
                                hipStream_t stream) {
  switch (op) {
    case kOpSum: return dispatch<kOpSum>(in, nullptr, out, nullptr, rows, width, width, 0.f, stream);
    case kOpMax: return dispatch<kOpMax>(in, nullptr, out, nullptr, rows, width, width, 0.f, stream);
    case kOpSoftmax: return dispatch<kOpSoftmax>(in, nullptr, out, nullptr, rows, width, width, 0.f, stream);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_rmsnorm(const float* in, const float* w, float* out, float* inv_rms, uint32_t tokens,
                          uint32_t width, uint32_t stride, float eps, hipStream_t stream) {
  return dispatch<kOpRms>(in, w, out, inv_rms, tokens, width, stride, eps, stream);
}

}  // namespace prom
