// FP32 products of few rows, C[m, n] = A[m, k] @ B[k, n] (+ R) with m <= 48: a
// decode step or a short prompt against a weight matrix.
//
// Such a product reads B once and does little else, so it is bound by HBM (or, for
// small B, by latency).  The macro tiles of sgemm_f32.hip run most of their rows as
// padding and stage B through LDS with a barrier per K tile, a chain of waits that
// a few workgroups per CU do not cover.  Here B goes from memory straight into the
// registers the matrix cores read it from, without LDS and without barriers:
//
//   * v_mfma_f32_16x16x4_f32 takes A[i][k] from lane i + 16 k and B[k][j] from lane
//     j + 16 k (k < 4).  A wave works on granules of 16 k: lane (g, i) loads four
//     consecutive k of A row i at k0 + 4 g, so in step c the lane groups hold
//     k = k0 + 4 g + c, and lane (g, j) loads kC consecutive columns of that row
//     of B (16 kC floats of a row per group); each of them feeds one MFMA;
//   * a workgroup owns 16 kC columns; its waves take the granules of its K slice in
//     turn and add their sums through LDS in a fixed order at the end (deterministic);
//   * where that leaves CUs idle K is also cut into slices over gridDim.y, whose
//     slabs a second kernel adds in slice order.
//
// Addresses go through buffer descriptors: rows of B past K and what lies past its
// end read zero, columns past n feed only outputs that are not stored, and rows of
// A past m are clamped to the last one (their outputs are not stored).  Any
// alignment of 4 bytes will do, so ragged operands need no padded copies.
#include <algorithm>
#include <cmath>

#include "reactor_internal.h"

namespace prom {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

struct RowsArgs {
  const float* a;
  const float* b;
  float* c;
  const float* r;
  int m, n, k;
  int lda, ldb, ldc, ldr;
  size_t slab;  // floats between the slices' slabs (gridDim.y > 1)
};

// The workgroup shapes: kC columns per lane, kW waves.
struct RowsShape {
  int c, w;
  double step, chain;  // us per granule of a full CU, and of one wave's chain
};

// Estimated time of a shape with S slices, from a least-squares fit (log time, rms
// 8 %) to 2004 runs at 60 products of 1 to 48 rows on MI355X, n 256..32768, k
// 512..16384.  A CU works through ceil(workgroups / 256) workgroups at `step` per
// granule (0.72 of it more per further 16 rows, the matrix cores' share), each wave
// through its own at `chain`, and B arrives at 6.2 TB/s at most.  The plan with the
// least estimate is within 4 % of the fastest measured on average, 27 % at worst
// (1x1418x4315); those runs' operands were in the caches.  us, the tiles of
// sgemm_f32.hip -> this, with B in the caches and, in brackets, with 1.2 GB of matrices in
// turn: 15x2048x1536 9.4 -> 5.5 (10.7 -> 10.5), 15x8192x2048 22.2 -> 11.9 (23.4 -> 15.0),
// 15x32768x2048 64.2 -> 40.9 (67.3 -> 49.7), 48x16384x8192 148 -> 118 (148 -> 118).
// Against a B that comes from HBM the estimate is low: by 9 % in the median of 160
// products, 26 % at the ninth decile.
constexpr RowsShape kShapes[] = {{1, 8, 0.0344, 0.305}, {1, 16, 0.0345, 0.491}, {2, 8, 0.0485, 0.385},
                                 {2, 16, 0.0512, 0.333}, {4, 4, 0.0916, 0.555}, {4, 8, 0.0897, 0.566}};
constexpr int kNumShapes = sizeof(kShapes) / sizeof(kShapes[0]);
constexpr double kMoreRows = 0.72, kLaunchUs = 3.97, kReduceUs = 3.12, kReduceBytesPerUs = 3.88e6,
                 kReadBytesPerUs = 6.18e6, kPartCu = 0.794;

double rows_us(const RowsShape& q, int splits, uint32_t m, uint32_t n, uint32_t k, int halves) {
  const long long groups = (long long)((n + 16 * q.c - 1) / (16 * q.c)) * splits;
  const int slice = ((int)((k + 15) / 16) + splits - 1) / splits;
  const double step = q.step * halves * (1.0 + kMoreRows * ((m + 15) / 16 - 1));
  const double rest = (double)(groups % 256);
  const double load = (double)(groups / 256) + (rest > 0 ? kPartCu + (1.0 - kPartCu) * rest / 256.0 : 0.0);
  const double run = std::max(load * slice * step, std::ceil((double)slice / q.w) * q.chain);
  const double read = (double)k * n * halves * 4.0 / kReadBytesPerUs;
  const double run2 = run * run, read2 = read * read;
  double us = kLaunchUs + std::sqrt(std::sqrt(run2 * run2 + read2 * read2));
  if (splits > 1) us += kReduceUs + (double)(splits + 1) * m * n * 4.0 / kReduceBytesPerUs;
  return us;
}

// kGe: B is [gate | up], n columns each; C = gelu_tanh(A @ gate) * (A @ up).
template <int kMB, int kC, int kW, bool kGe>
__global__ __launch_bounds__(64 * kW) void sgemm_rows_kernel(const RowsArgs p) {
  constexpr int kH = kGe ? 2 : 1;         // column halves: gate and up
  constexpr int kCols = 16 * kC;          // columns of a half
  constexpr int kBlock = 16 * kMB * kCols * kH;  // floats of a workgroup's sums
  __shared__ float sums[kW][kBlock];
  const int tid = (int)threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = lane >> 4, li = lane & 15;
  const int col0 = xcd_pid((int)blockIdx.x, (int)gridDim.x) * kCols;
  const int all = (p.k + 15) / 16;
  const int g0 = (int)((long long)blockIdx.y * all / gridDim.y);
  const int g1 = (int)((long long)(blockIdx.y + 1) * all / gridDim.y);

  const __amdgpu_buffer_rsrc_t ra =
      __builtin_amdgcn_make_buffer_rsrc((void*)p.a, (short)0, (int)(((size_t)(p.m - 1) * p.lda + p.k) * 4), 0x00020000);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
      (void*)p.b, (short)0, (int)(((size_t)(p.k - 1) * p.ldb + (size_t)p.n * kH) * 4), 0x00020000);
  uint32_t a_off[kMB];
#pragma unroll
  for (int mb = 0; mb < kMB; ++mb) a_off[mb] = (uint32_t)((min(16 * mb + li, p.m - 1) * p.lda + 4 * grp) * 4);
  const uint32_t b_off = (uint32_t)((4 * grp * p.ldb + col0 + kC * li) * 4);
  const uint32_t row = (uint32_t)p.ldb * 4u;

  struct Granule {
    floatx4 a[kMB];
    float b[kH][4][kC];
  };
  auto load = [&](Granule& q, int g) __attribute__((always_inline)) {
    const int k0 = 16 * g;
#pragma unroll
    for (int h = 0; h < kH; ++h)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const uint32_t off = b_off + (uint32_t)(k0 + c) * row + (uint32_t)(h * p.n) * 4u;
        if constexpr (kC == 4) {
          const floatx4 v = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rb, off, 0, 0));
#pragma unroll
          for (int j = 0; j < 4; ++j) q.b[h][c][j] = v[j];
        } else if constexpr (kC == 2) {
          const float2 v = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(rb, off, 0, 0));
          q.b[h][c][0] = v.x;
          q.b[h][c][1] = v.y;
        } else {
          q.b[h][c][0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rb, off, 0, 0));
        }
      }
#pragma unroll
    for (int mb = 0; mb < kMB; ++mb)
      q.a[mb] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(ra, a_off[mb] + 4u * k0, 0, 0));
    if (k0 + 16 > p.k) {  // the last granule of a ragged k: A past k is another row's
#pragma unroll
      for (int mb = 0; mb < kMB; ++mb)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (k0 + 4 * grp + c >= p.k) q.a[mb][c] = 0.0f;
    }
  };
  // Sums of two granules (32 of k) at a time go into `total`: a chain of 32 and one of
  // the blocks, whose rounding is that of the tiles' K slices or less where one chain
  // over a long K has more (13x9344x7680: 5.6e-7 of the result, the tiles 3.3e-7).
  floatx4 acc[kH][kMB][kC], total[kH][kMB][kC];
#pragma unroll
  for (int h = 0; h < kH; ++h)
#pragma unroll
    for (int mb = 0; mb < kMB; ++mb)
#pragma unroll
      for (int j = 0; j < kC; ++j) acc[h][mb][j] = total[h][mb][j] = floatx4{};
  auto add_up = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < kH; ++h)
#pragma unroll
      for (int mb = 0; mb < kMB; ++mb)
#pragma unroll
        for (int j = 0; j < kC; ++j) {
          total[h][mb][j] += acc[h][mb][j];
          acc[h][mb][j] = floatx4{};
        }
  };
  auto compute = [&](const Granule& q) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int h = 0; h < kH; ++h)
#pragma unroll
        for (int j = 0; j < kC; ++j)
#pragma unroll
          for (int mb = 0; mb < kMB; ++mb)
            acc[h][mb][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(q.a[mb][c], q.b[h][c][j], acc[h][mb][j], 0, 0, 0);
  };

  // The wave's granules are g0 + wave, then every kW-th; the next one's loads are in
  // flight while one is multiplied (two ahead measured 0 to 5 % slower at nine products,
  // with B in the caches and from HBM alike: the other waves of the CU cover the rest).
  Granule q;
  int g = g0 + wave;
  if (g < g1) load(q, g);
  for (int done = 1; g + kW < g1; g += kW, ++done) {
    Granule next;
    load(next, g + kW);
    compute(q);
    if ((done & 1) == 0) add_up();
    q = next;
  }
  if (g < g1) compute(q);
  add_up();

  // D[i][j] is in lane j + 16 (i / 4), register i % 4; block j of a half holds its
  // columns kC * (lane % 16) + j.
#pragma unroll
  for (int h = 0; h < kH; ++h)
#pragma unroll
    for (int mb = 0; mb < kMB; ++mb)
#pragma unroll
      for (int j = 0; j < kC; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          sums[wave][((h * 16 * kMB) + 16 * mb + 4 * grp + i) * kCols + kC * li + j] = total[h][mb][j][i];
  __syncthreads();
  // The waves' sums, added in pairs: log2(kW) roundings each, in a fixed order.
  auto sum_waves = [&](int e) __attribute__((always_inline)) {
    float v[kW];
#pragma unroll
    for (int w = 0; w < kW; ++w) v[w] = sums[w][e];
#pragma unroll
    for (int step = kW / 2; step > 0; step /= 2)
#pragma unroll
      for (int w = 0; w < step; ++w) v[w] += v[w + step];
    return v[0];
  };
  float* out = p.c + (gridDim.y > 1 ? blockIdx.y * p.slab : 0);
  for (int e = tid; e < 16 * kMB * kCols; e += 64 * kW) {
    const int i = e / kCols, col = col0 + e % kCols;
    float v = sum_waves(e);
    if constexpr (kGe) v = gelu_tanh(v) * sum_waves(e + kBlock / 2);
    if (i < p.m && col < p.n) {
      if (p.r != nullptr) v += p.r[(size_t)i * p.ldr + col];
      out[(size_t)i * p.ldc + col] = v;
    }
  }
}

template <int kMB, bool kGe>
hipError_t launch_shape(int shape, dim3 grid, const RowsArgs& p, hipStream_t stream) {
#define ROWS(I, C, W)                                                                                        \
  case I:                                                                                                    \
    hipLaunchKernelGGL((sgemm_rows_kernel<kMB, C, W, kGe>), grid, dim3(64 * W), 0, stream, p);               \
    break
  switch (shape) {
    ROWS(0, 1, 8);
    ROWS(1, 1, 16);
    ROWS(2, 2, 8);
    default:
      if constexpr (kGe) {
        return hipErrorInvalidValue;
      } else {
        switch (shape) {
          ROWS(3, 2, 16);
          ROWS(4, 4, 4);
          ROWS(5, 4, 8);
          default:
            return hipErrorInvalidValue;
        }
      }
  }
#undef ROWS
  return hipGetLastError();
}

template <bool kGe>
hipError_t launch_rows_of(int shape, int splits, const RowsArgs& p, hipStream_t stream) {
  const unsigned cols = 16u * (unsigned)kShapes[shape].c;
  const dim3 grid(((unsigned)p.n + cols - 1) / cols, (unsigned)splits);
  switch ((p.m + 15) / 16) {
    case 1: return launch_shape<1, kGe>(shape, grid, p, stream);
    case 2: return launch_shape<2, kGe>(shape, grid, p, stream);
    case 3: return launch_shape<3, kGe>(shape, grid, p, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

bool sgemm_rows_take(uint32_t m, uint32_t k, int lda, int ldb) {
  const size_t lim = (1ull << 31) - (1u << 16);
  return m <= 48u && (size_t)m * lda * 4 < lim && ((size_t)k + 32) * ldb * 4 < lim;
}

SgemmRowsPlan plan_sgemm_rows(uint32_t m, uint32_t n, uint32_t k, bool geglu, uint64_t max_partial_floats) {
  static const int kSplits[] = {1, 2, 3, 4, 6, 8, 12, 16};
  SgemmRowsPlan best{0, 1, 1e300};
  for (int i = 0; i < (geglu ? 3 : kNumShapes); ++i) {
    for (int s : kSplits) {
      if (s > 1 && (geglu || (int)((k + 15) / 16) < s * kShapes[i].w || (uint64_t)s * m * n > max_partial_floats))
        break;
      const double us = rows_us(kShapes[i], s, m, n, k, geglu ? 2 : 1);
      if (us < best.us) best = SgemmRowsPlan{i, s, us};
    }
  }
  return best;
}

int sgemm_rows_columns(const SgemmRowsPlan& plan) { return 16 * kShapes[plan.shape].c; }

hipError_t launch_sgemm_rows(const SgemmRowsPlan& plan, const float* a, int lda, const float* b, int ldb, float* c,
                             int ldc, uint32_t m, uint32_t n, uint32_t k, const float* residual, int ldr,
                             hipStream_t stream) {
  const RowsArgs p{a, b, c, residual, (int)m, (int)n, (int)k, lda, ldb, ldc, ldr, (size_t)m * ldc};
  return launch_rows_of<false>(plan.shape, plan.splits, p, stream);
}

hipError_t launch_sgemm_rows_geglu(const SgemmRowsPlan& plan, const float* a, int lda, const float* w, float* h,
                                   int ldh, uint32_t m, uint32_t f, uint32_t k, hipStream_t stream) {
  const RowsArgs p{a, w, h, nullptr, (int)m, (int)f, (int)k, lda, (int)(2 * f), ldh, 0, 0};
  return launch_rows_of<true>(plan.shape, 1, p, stream);
}

}  // namespace prom
