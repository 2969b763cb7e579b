// bf16 GEMM kernels for the shapes the 256x256 kernel (gemm_bf16.hip) does not
// fill the chip with: few rows, few tiles, K tails, ragged sizes.
//
// One template, instantiated at several macro tiles.  A workgroup's waves form
// a kWM x kWN grid, each owning kMI x kNI MFMA 32x32x16 blocks.  A and B tiles
// travel HBM -> LDS by buffer_load ... lds (16 bytes per lane, 1 KiB per
// instruction) into a ring of kSt stages; LDS keeps A [m][k] and B [k][n] as
// they lie in memory, the B operand comes from transpose reads.  Chunk (16
// bytes) positions are XOR-swizzled by row so that operand reads are free of
// bank conflicts; the swizzle is applied by the source address of each lane.
//
// Every transfer goes through a descriptor that is advanced to the tile's
// first byte and whose range ends at the operand's end, so rows past M or K
// and columns past the end read zero; A's columns past K in the last tile are
// sent out of range, so a K tail adds exact zeros.  Only 16-byte alignment
// (base, lda, ldb; k a multiple of 8) is asked of the operands; others are first
// copied to zero-padded buffers.
//
// K is cut into `splits` slices over gridDim.y; each slice writes fp32 sums to
// its slab and a second kernel adds the slabs in slice order (deterministic).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "reactor_internal.h"

namespace prom {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef int int4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

constexpr int kGroupM = 8;
constexpr uint32_t kOutOfRange = 0x80000000u;  // past every descriptor range

__device__ __forceinline__ uint16_t to_bf16_rne(float v) {
  const uint32_t bits = __float_as_uint(v);
  return (uint16_t)((bits + 0x7FFFu + ((bits >> 16) & 1u)) >> 16);
}

struct Bf16Args {
  const uint16_t* a;
  const uint16_t* b;
  float* c;          // fp32 output, or the slabs of a K split
  uint16_t* cb;      // bf16 output when not null
  const float* r;    // residual, may be null
  int m, n, k;
  int lda, ldb, ldc, ldr;
  int tiles_m, tiles_n;
  size_t slab;       // floats between slabs (K split only)
};

template <int kMI_, int kNI_, int kWM_, int kWN_, int kBK_, int kSt_, bool kPre_ = false>
struct Cfg {
  static constexpr bool kPre = kPre_;
  static constexpr int kMI = kMI_, kNI = kNI_, kWM = kWM_, kWN = kWN_, kBK = kBK_, kSt = kSt_;
  static constexpr int kWaves = kWM * kWN;
  static constexpr int kBM = 32 * kMI * kWM, kBN = 32 * kNI * kWN;
  static constexpr int kABytes = kBM * kBK * 2, kBBytes = kBK * kBN * 2;
  static constexpr int kStage = kABytes + kBBytes;
  static constexpr int kAX = kABytes / 1024 / kWaves, kBX = kBBytes / 1024 / kWaves;  // transfers per wave and tile
  static constexpr int kX = kAX + kBX;
  static_assert(kAX * 1024 * kWaves == kABytes && kBX * 1024 * kWaves == kBBytes, "whole transfers per wave");
  static_assert(kSt >= (kPre ? 3 : 2) && kSt * kStage <= 163840 && (kSt - 2) * kX < 64, "ring");
};

// Position of A chunk c of row r (rows of kBK values), and of B chunk c of row k.
template <int kBK>
__device__ __forceinline__ int swz_a(int r) {
  return kBK == 32 ? ((r >> 2) & 3) : ((r & 7) ^ ((r >> 3) & 1));
}
template <int kBN>
__device__ __forceinline__ int swz_b(int k) {
  if constexpr (kBN == 256) return (0xEA40 >> (4 * (k & 3))) & 15;
  if constexpr (kBN == 128) return 4 * (k & 3);
  return 4 * ((k >> 1) & 1);
}

template <int kN>
__device__ __forceinline__ void wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kN) : "memory");
}

// At most min(kMost, n) tiles of kX transfers may stay in flight.
template <int kX, int kMost>
__device__ __forceinline__ void wait_tiles(int n) {
  if constexpr (kMost > 0) {
    if (n < kMost) {
      wait_tiles<kX, kMost - 1>(n);
      return;
    }
  }
  wait_vmcnt<kX * kMost>();
}

// kSwiGLU: B is [K, 2N] = [gate | up]; a wave's two 32-column blocks are a gate
// block and its up block (kNI == 2) and the output is silu(gate) * up, N
// columns in bf16.
template <class C, bool kSwiGLU>
__global__ __launch_bounds__(64 * C::kWaves, 2) void gemm_bf16_tile_kernel(const Bf16Args g) {
  static_assert(!kSwiGLU || C::kNI == 2, "gate and up blocks of a wave");
  __shared__ __attribute__((aligned(1024))) char lds[C::kSt * C::kStage];
  constexpr int kBK = C::kBK, kBN = C::kBN, kSteps = kBK / 16;
  const int num_tiles = g.tiles_m * g.tiles_n;
  int tm, tn;
  {
    const int pid = xcd_pid((int)blockIdx.x, num_tiles);
    const int per_group = kGroupM * g.tiles_n;
    const int group = pid / per_group;
    const int first_m = group * kGroupM;
    const int group_m = min(g.tiles_m - first_m, kGroupM);
    const int in_group = pid - group * per_group;
    tm = first_m + in_group % group_m;
    tn = in_group / group_m;
  }
  const int row0 = tm * C::kBM;
  const int col0 = kSwiGLU ? tn * (kBN / 2) : tn * kBN;
  const int all_tiles = (g.k + kBK - 1) / kBK;
  const int splits = (int)gridDim.y;
  const int kt0 = (int)((long long)blockIdx.y * all_tiles / splits);
  const int kn = (int)((long long)(blockIdx.y + 1) * all_tiles / splits) - kt0;

  const int tid = (int)threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / C::kWN, wn = wave % C::kWN;

  // This wave's transfers: A block q (1 KiB: 512 / kBK rows) and B block q (512 / kBN
  // rows), q = wave * kAX + i.  Offsets are relative to the tile's first byte.
  uint32_t a_off[C::kAX], b_off[C::kBX];
  constexpr int kAChunks = kBK / 8, kBChunks = kBN / 8;
  auto a_rc = [&](int i, int* r, int* c) {
    const int e = 64 * (wave * C::kAX + i) + lane;
    *r = e / kAChunks;
    *c = (e % kAChunks) ^ swz_a<kBK>(*r);
  };
#pragma unroll
  for (int i = 0; i < C::kAX; ++i) {
    int r, c;
    a_rc(i, &r, &c);
    a_off[i] = (uint32_t)((r * g.lda + 8 * c) * 2);
  }
#pragma unroll
  for (int i = 0; i < C::kBX; ++i) {
    const int e = 64 * (wave * C::kBX + i) + lane;
    const int kr = e / kBChunks;
    const int cb = (e % kBChunks) ^ swz_b<kBN>(kr);
    int col = 8 * cb;
    if constexpr (kSwiGLU) col = (col >> 6) * 32 + (col & 31) + ((col & 32) ? g.n : 0);
    b_off[i] = (uint32_t)((kr * g.ldb + col) * 2);
  }
  // First byte and remaining bytes of the next tile to issue, per operand.
  // (K and the columns rounded up to whole 16-byte chunks: a padded copy's tail.)
  const int k8 = (g.k + 7) & ~7, n8 = ((kSwiGLU ? 2 * g.n : g.n) + 7) & ~7;
  const char* a_ptr = (const char*)(g.a + (size_t)row0 * g.lda + (size_t)kt0 * kBK);
  long long a_left = ((long long)(g.m - 1 - row0) * g.lda + k8 - (long long)kt0 * kBK) * 2;
  const char* b_ptr = (const char*)(g.b + (size_t)kt0 * kBK * g.ldb + col0);
  long long b_left = ((long long)(g.k - 1 - kt0 * kBK) * g.ldb + n8 - col0) * 2;
  const long long b_step = (long long)kBK * g.ldb * 2;
  int issued = 0;
  auto desc = [](const char* p, long long left) {
    const unsigned long long a = (unsigned long long)p;
    const unsigned range = left < 0 ? 0u : (left > 0x7fffffffll ? 0x7fffffffu : (unsigned)left);
    int4v d;
    d.x = __builtin_amdgcn_readfirstlane((int)(a & 0xffffffffu));
    d.y = __builtin_amdgcn_readfirstlane((int)(a >> 32));
    d.z = __builtin_amdgcn_readfirstlane((int)range);
    d.w = 0x00020000;
    return d;
  };
  const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)lds;
  int4v da = desc(a_ptr, a_left), db = desc(b_ptr, b_left);
  uint32_t fill = lds0;  // LDS address of the stage the next tile goes to
  // Transfer j (0 .. kX-1) of the tile being issued; tail: its last chunks lie past K.
  auto issue_one = [&](int j, bool tail) __attribute__((always_inline)) {
    if (j < C::kAX) {
      uint32_t off = a_off[j];
      if (tail) {
        int r, c;
        a_rc(j, &r, &c);
        if ((kt0 + issued) * kBK + 8 * c >= g.k) off = kOutOfRange;
      }
      const uint32_t to = __builtin_amdgcn_readfirstlane(fill + (wave * C::kAX + j) * 1024);
      asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(to), "v"(off), "s"(da)
                   : "memory", "m0");
    } else {
      const uint32_t to =
          __builtin_amdgcn_readfirstlane(fill + C::kABytes + (wave * C::kBX + (j - C::kAX)) * 1024);
      asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(to), "v"(b_off[j - C::kAX]),
                   "s"(db)
                   : "memory", "m0");
    }
  };
  auto advance = [&]() __attribute__((always_inline)) {
    a_ptr += kBK * 2;
    a_left -= kBK * 2;
    b_ptr += b_step;
    b_left -= b_step;
    da = desc(a_ptr, a_left);
    db = desc(b_ptr, b_left);
    fill = fill + C::kStage == lds0 + C::kSt * C::kStage ? lds0 : fill + C::kStage;
    ++issued;
  };

  const int lrow = lane & 31;
  const int hk = lane >> 5;
  const int tr_row = 8 * hk + ((lane & 15) >> 2);
  const int tr_e = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  // Byte offsets within a stage.  A rows 32 mi further down share the swizzle, and
  // chunk 2s + hk of a row is chunk hk's position XOR 2s; B rows 16 s further share
  // theirs too, so s and mi (A) or s (B) are immediate offsets of the reads.
  const int r0 = wm * C::kMI * 32 + lrow;
  uint32_t a_base[kSteps], b_base[C::kNI];
#pragma unroll
  for (int s = 0; s < kSteps; ++s) a_base[s] = (uint32_t)(r0 * kBK * 2 + (((2 * s + hk) ^ swz_a<kBK>(r0)) << 4));
#pragma unroll
  for (int ni = 0; ni < C::kNI; ++ni) {
    const int col = (wn * C::kNI + ni) * 32 + tr_e;
    b_base[ni] = (uint32_t)(C::kABytes + tr_row * kBN * 2 + (((col >> 3) ^ swz_b<kBN>(tr_row)) << 4) + (col & 7) * 2);
  }
  struct Frags {
    bf16x8 a[C::kMI], b[C::kNI];
  };
  auto read = [&](uint32_t st, int s) __attribute__((always_inline)) {
    Frags f;
    const char* pa = lds + (st + a_base[s]);
#pragma unroll
    for (int mi = 0; mi < C::kMI; ++mi) f.a[mi] = *reinterpret_cast<const bf16x8*>(pa + mi * 32 * kBK * 2);
#pragma unroll
    for (int ni = 0; ni < C::kNI; ++ni) {
      const char* pb = lds + (st + b_base[ni]) + s * 16 * kBN * 2;
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)pb);
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(pb + 4 * kBN * 2));
      f.b[ni] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
    return f;
  };

  floatx16 acc[C::kMI][C::kNI];
#pragma unroll
  for (int i = 0; i < C::kMI; ++i)
#pragma unroll
    for (int j = 0; j < C::kNI; ++j) acc[i][j] = floatx16{};

  // Tiles of this slice whose A chunks all lie below K: all, or all but the last.
  const int whole = kn - ((kt0 + kn) * kBK > g.k ? 1 : 0);
#pragma unroll
  for (int s = 0; s < C::kSt - 1; ++s)
    if (s < kn) {
#pragma unroll
      for (int j = 0; j < C::kX; ++j) issue_one(j, s >= whole);
      advance();
    }
  // kPre: tile t+1 has landed before tile t's MFMAs end, so its first operands
  // are read ahead of the next barrier (one stage less stays in flight).
  constexpr int kDepth = C::kPre ? C::kSt - 3 : C::kSt - 2;
  auto barrier = [] {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  uint32_t cur = 0;
  Frags f;
  if constexpr (C::kPre) {
    wait_tiles<C::kX, C::kSt - 2>(kn - 1);
    barrier();
    f = read(0, 0);
  }
  // Step t: tile t (kPre: t+1) has landed for this wave, later ones may stay in
  // flight; after the barrier it is complete for all waves and tile t-1's stage is
  // free.  The transfers of tile t + kSt - 1 go out between the MFMAs, spread evenly.
  auto step = [&](int t, auto more_c, auto tail_c) __attribute__((always_inline)) {
    constexpr bool kMore = decltype(more_c)::value, kTail = decltype(tail_c)::value;
    constexpr int kMfma = kSteps * C::kMI * C::kNI;
    if constexpr (kMore && !kTail)
      wait_vmcnt<C::kX * kDepth>();
    else
      wait_tiles<C::kX, kDepth>(kn - 1 - t - (C::kPre ? 1 : 0));
    barrier();
    const uint32_t next = cur + C::kStage == C::kSt * C::kStage ? 0 : cur + C::kStage;
    if constexpr (!C::kPre) f = read(cur, 0);
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      Frags nf;
      if (s + 1 < kSteps) nf = read(cur, s + 1);
      __builtin_amdgcn_sched_barrier(0);  // the next step's reads go out before this one's MFMAs
#pragma unroll
      for (int mi = 0; mi < C::kMI; ++mi)
#pragma unroll
        for (int ni = 0; ni < C::kNI; ++ni) {
          const int at = (s * C::kMI + mi) * C::kNI + ni;
          acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[mi], f.b[ni], acc[mi][ni], 0, 0, 0);
#pragma unroll
          for (int j = 0; j < C::kX; ++j)
            if (kMore && j * kMfma / C::kX == at) issue_one(j, kTail);
        }
      if (s + 1 < kSteps) f = nf;
    }
    if constexpr (kMore) advance();
    if constexpr (C::kPre)
      if (kMore || t + 1 < kn) f = read(next, 0);
    cur = next;
  };
  const std::integral_constant<bool, true> yes{};
  const std::integral_constant<bool, false> no{};
  int t = 0;
  for (; t + C::kSt - 1 < whole; ++t) step(t, yes, no);
  if (t + C::kSt - 1 < kn) {
    step(t, yes, yes);
    ++t;
  }
  for (; t < kn; ++t) step(t, no, no);

  // Accumulator layout: lane l, register r holds row 8 (r/4) + 4 (l/32) + r%4, column l%32.
  const int lgrp = hk * 4;
  if constexpr (kSwiGLU) {
    const int col = col0 + wn * 32 + lrow;
    if (col >= g.n) return;
#pragma unroll
    for (int mi = 0; mi < C::kMI; ++mi) {
      const int rb = row0 + (wm * C::kMI + mi) * 32 + lgrp;
      uint16_t* hp = g.cb + (size_t)rb * g.ldc + col;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int dr = 8 * (r >> 2) + (r & 3);
        if (rb + dr < g.m) hp[(size_t)dr * g.ldc] = to_bf16_rne(silu_mul(acc[mi][0][r], acc[mi][1][r]));
      }
    }
    return;
  }
#pragma unroll
  for (int mi = 0; mi < C::kMI; ++mi)
#pragma unroll
    for (int ni = 0; ni < C::kNI; ++ni) {
      const int col = col0 + (wn * C::kNI + ni) * 32 + lrow;
      if (col >= g.n) continue;
      const int rb = row0 + (wm * C::kMI + mi) * 32 + lgrp;
      if (splits > 1) {
        float* cp = g.c + blockIdx.y * g.slab + (size_t)rb * g.ldc + col;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int dr = 8 * (r >> 2) + (r & 3);
          if (rb + dr < g.m) cp[(size_t)dr * g.ldc] = acc[mi][ni][r];
        }
        continue;
      }
      const float* rp = g.r != nullptr ? g.r + (size_t)rb * g.ldr + col : nullptr;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int dr = 8 * (r >> 2) + (r & 3);
        if (rb + dr < g.m) {
          float v = acc[mi][ni][r];
          if (rp != nullptr) v += rp[(size_t)dr * g.ldr];
          if (g.cb != nullptr)
            g.cb[(size_t)(rb + dr) * g.ldc + col] = to_bf16_rne(v);
          else
            g.c[(size_t)(rb + dr) * g.ldc + col] = v;
        }
      }
    }
}

// C = sum over slabs (slice order) + R, four columns per thread; slab pitch n4
// (a multiple of 4).
__global__ __launch_bounds__(256) void bf16_splitk_reduce_kernel(const float* __restrict__ p, size_t slab, int splits,
                                                                 int n4, float* c, uint16_t* cb, int ldc,
                                                                 const float* r, int ldr, int m, int n, int vec) {
  const int c4 = (int)(blockIdx.x * 64 + (threadIdx.x & 63));
  const int col = 4 * c4;
  if (col >= n) return;
  for (int row = (int)(blockIdx.y * 4 + (threadIdx.x >> 6)); row < m; row += (int)gridDim.y * 4) {
    const float* src = p + (size_t)row * n4 + col;
    floatx4 v = *reinterpret_cast<const floatx4*>(src);
    int s = 1;
    for (; s + 3 < splits; s += 4) {  // four slabs' loads in flight, added in order
      const floatx4 a = *reinterpret_cast<const floatx4*>(src + s * slab);
      const floatx4 b = *reinterpret_cast<const floatx4*>(src + (s + 1) * slab);
      const floatx4 d = *reinterpret_cast<const floatx4*>(src + (s + 2) * slab);
      const floatx4 e = *reinterpret_cast<const floatx4*>(src + (s + 3) * slab);
      v = v + a;
      v = v + b;
      v = v + d;
      v = v + e;
    }
    for (; s < splits; ++s) v = v + *reinterpret_cast<const floatx4*>(src + s * slab);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (r != nullptr && col + j < n) v[j] += r[(size_t)row * ldr + col + j];
    if (vec) {
      if (cb != nullptr) {
        const uint32_t lo = to_bf16_rne(v.x) | ((uint32_t)to_bf16_rne(v.y) << 16);
        const uint32_t hi = to_bf16_rne(v.z) | ((uint32_t)to_bf16_rne(v.w) << 16);
        *reinterpret_cast<uint2*>(cb + (size_t)row * ldc + col) = make_uint2(lo, hi);
      } else {
        *reinterpret_cast<floatx4*>(c + (size_t)row * ldc + col) = v;
      }
      continue;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (col + j >= n) break;
      if (cb != nullptr)
        cb[(size_t)row * ldc + col + j] = to_bf16_rne(v[j]);
      else
        c[(size_t)row * ldc + col + j] = v[j];
    }
  }
}

// The macro tiles.  K tiles are 64 wide: a row of A is then a whole 128-byte
// line (with 32-wide K tiles, half lines, the 64x128 and 128x256 tiles ran 20 %
// slower).  The first three run two workgroups per CU, the others one.
#define BF16_TILES(X)                          \
  X(0, 1, 1, 1, 4, 64, 4)       /* 32x128 */   \
  X(1, 1, 1, 2, 2, 64, 5)       /* 64x64 */    \
  X(2, 1, 2, 2, 2, 64, 3)       /* 64x128 */   \
  X(3, 1, 2, 2, 4, 64, 4)       /* 64x256 */   \
  X(4, 1, 2, 4, 2, 64, 4)       /* 128x128 */  \
  X(5, 3, 1, 2, 4, 64, 4, true) /* 192x128 */  \
  X(6, 2, 2, 2, 4, 64, 3)       /* 128x256 */  \
  X(7, 3, 2, 2, 4, 64, 2)       /* 192x256 */  \
  X(8, 4, 2, 2, 4, 64, 2)       /* 256x256 */

struct TileInfo {
  int bm, bn, threads, ni;
};
#define X(i, ...) \
  {Cfg<__VA_ARGS__>::kBM, Cfg<__VA_ARGS__>::kBN, 64 * Cfg<__VA_ARGS__>::kWaves, Cfg<__VA_ARGS__>::kNI},
constexpr TileInfo kTiles[] = {BF16_TILES(X)};
#undef X
constexpr int kNumTiles = sizeof(kTiles) / sizeof(kTiles[0]);
constexpr int kTileK = 64;

// Estimated microseconds of W workgroups of tile t, kt K tiles of 64 each: the
// CUs are filled in rounds of 256 * occ; a round of w workgroups per CU takes
// `fill` (prologue and epilogue) plus kt times step[w-1]; in a last round that
// does not fill the chip the step falls towards `idle` of it.  The constants are
// a least-squares fit (log time) to 1859 (tile, K slices) runs at 58 shapes on
// MI355X, m 32..4224, n 256..11520, k 256..10240: rms 4.4 %, and the plan with
// the least estimate is within 2 % of the fastest measured on average, 15 % at worst.
// A large B (past what the caches hold) is read at the rate its bytes in flight
// allow: `flight` KiB per workgroup over ~1.5 us of latency, 5 TB/s at most
// (32x11520x10240, one K slice of 64x64 tiles 72 us, four of 64x256 46 us).
struct TileCost {
  int occ;
  double step[2], fill, idle, flight;
};
constexpr TileCost kCost[kNumTiles + 1] = {
    {2, {0.203, 0.452}, 2.36, 0.86, 48},  // 32x128
    {2, {0.190, 0.375}, 2.49, 0.77, 32},  // 64x64
    {2, {0.325, 0.648}, 2.84, 0.58, 32},  // 64x128
    {1, {0.639, 0.639}, 3.49, 0.41, 96},  // 64x256
    {1, {0.585, 0.585}, 3.49, 0.46, 48},  // 128x128
    {1, {0.740, 0.740}, 5.24, 0.36, 32},  // 192x128
    {1, {0.945, 0.945}, 5.67, 0.42, 64},  // 128x256
    {1, {1.529, 1.529}, 6.57, 0.49, 32},  // 192x256
    {1, {1.852, 1.852}, 8.60, 0.46, 32},  // 256x256
    {1, {1.720, 1.720}, 9.10, 0.46, 64},  // the five-stage 256x256 kernel (gemm_bf16.hip)
};
constexpr double kLaunchUs = 3.9, kReduceUs = 2.2, kReduceBytesPerUs = 10.0e6, kReadBytesPerUs = 5.0e6;
constexpr double kLargeB = 5.0e7, kLatencyUs = 1.5;

double rounds_us(int t, long long w_total, int kt) {
  const TileCost& c = kCost[t];
  const long long slots = 256ll * c.occ;
  const long long full = w_total / slots, rest = w_total - full * slots;
  double us = (double)full * (c.fill + kt * c.step[c.occ - 1]);
  if (rest > 0) {
    const int w = (int)((rest + 255) / 256);
    us += c.fill + kt * c.step[w - 1] * (c.idle + (1.0 - c.idle) * (double)rest / (256.0 * w));
  }
  return us;
}

hipError_t launch_tile(int tile, int splits, bool swiglu, const Bf16Args& g, hipStream_t stream) {
  const dim3 grid((unsigned)(g.tiles_m * g.tiles_n), (unsigned)splits);
  const dim3 block((unsigned)kTiles[tile].threads);
  if (swiglu) {
    switch (tile) {
#define X(i, ...)                                                                                             \
  case i:                                                                                                     \
    if constexpr (Cfg<__VA_ARGS__>::kNI == 2)                                                                 \
      hipLaunchKernelGGL((gemm_bf16_tile_kernel<Cfg<__VA_ARGS__>, true>), grid, block, 0, stream, g);         \
    else                                                                                                      \
      return hipErrorInvalidValue;                                                                            \
    break;
      BF16_TILES(X)
#undef X
    }
    return hipGetLastError();
  }
  switch (tile) {
#define X(i, ...)                                                                                      \
  case i:                                                                                              \
    hipLaunchKernelGGL((gemm_bf16_tile_kernel<Cfg<__VA_ARGS__>, false>), grid, block, 0, stream, g);   \
    break;
    BF16_TILES(X)
#undef X
  }
  return hipGetLastError();
}

// Every 32-bit offset of a tile stays below 2^31: 256 rows of A, 64 rows of B.
bool tiles_in_range(int lda, int ldb) { return (size_t)lda < (1u << 22) && (size_t)ldb < (1u << 23); }

}  // namespace

double bf16_five_stage_us(uint32_t m, uint32_t n, uint32_t k, int tail_splits) {
  const long long tiles = (long long)((m + 255) / 256) * ((n + 255) / 256);
  const int kt = (int)((k + kTileK - 1) / kTileK);
  if (tail_splits < 2) return kLaunchUs + rounds_us(kNumTiles, tiles, kt);
  const long long rest = tiles % 256;
  return kLaunchUs + rounds_us(kNumTiles, tiles - rest, kt) +
         rounds_us(kNumTiles, rest * tail_splits, (kt + tail_splits - 1) / tail_splits) + kLaunchUs + 5.0;
}

Bf16TilePlan plan_bf16_tiles(uint32_t m, uint32_t n, uint32_t k, bool swiglu) {
  static const int kSplits[] = {1, 2, 3, 4, 6, 8, 12, 16};
  const double read_us = 2.0 * ((double)m * k + (double)k * n) / kReadBytesPerUs;
  const int all = (int)((k + kTileK - 1) / kTileK);
  Bf16TilePlan best{0, 1, 1e300};
  for (int t = 0; t < kNumTiles; ++t) {
    if (swiglu && kTiles[t].ni != 2) continue;
    const long long tiles =
        (long long)((m + kTiles[t].bm - 1) / kTiles[t].bm) * ((n + kTiles[t].bn - 1) / kTiles[t].bn);
    for (int s : kSplits) {
      if (s > 1 && (swiglu || all < 3 * s)) break;
      double us = std::max(read_us, rounds_us(t, tiles * s, (all + s - 1) / s));
      if (2.0 * k * n > kLargeB) {
        const double readers = (double)std::min<long long>(tiles * s, 256ll * kCost[t].occ) /
                               ((m + kTiles[t].bm - 1) / kTiles[t].bm);
        const double rate = std::min(kReadBytesPerUs, readers * kCost[t].flight * 1024.0 / kLatencyUs);
        us = std::max(us, kCost[t].fill + 2.0 * k * n / rate);
      }
      us += kLaunchUs;
      if (s > 1) us += kReduceUs + (double)(s + 1) * m * n * 4.0 / kReduceBytesPerUs;
      if (us < best.us) best = Bf16TilePlan{t, s, us};
    }
  }
  return best;
}

static_assert(kNumTiles == (int)kBf16FiveStage, "the kernels' numbers");

bool bf16_tile_has_swiglu(uint32_t tile) { return tile < (uint32_t)kNumTiles && kTiles[tile].ni == 2; }

bool bf16_tiles_take(const uint16_t* a, int lda, const uint16_t* b, int ldb, uint32_t k) {
  return k % 8 == 0 && lda % 8 == 0 && ldb % 8 == 0 && ((uintptr_t)a & 15u) == 0 && ((uintptr_t)b & 15u) == 0 &&
         tiles_in_range(lda, ldb);
}

hipError_t launch_bf16_tiles(Bf16TilePlan p, bool swiglu, const uint16_t* a, int lda, const uint16_t* b, int ldb,
                             float* c, uint16_t* cb, int ldc, uint32_t m, uint32_t n, uint32_t k,
                             const float* residual, int ldr, hipStream_t stream) {
  const TileInfo& ti = kTiles[p.tile];
  Bf16Args g{};
  g.a = a;
  g.b = b;
  g.m = (int)m;
  g.n = (int)n;
  g.k = (int)k;
  g.lda = lda;
  g.ldb = ldb;
  g.tiles_m = (int)((m + ti.bm - 1) / ti.bm);
  const uint32_t cols = swiglu ? ti.bn / 2 : ti.bn;
  g.tiles_n = (int)((n + cols - 1) / cols);
  float* part = nullptr;
  const uint32_t n4 = (n + 3u) & ~3u;
  if (p.splits > 1) {
    part = static_cast<float*>(staging(6, (size_t)p.splits * m * n4 * sizeof(float)));
    if (part == nullptr) p.splits = 1;
  }
  if (p.splits == 1) {
    g.c = c;
    g.cb = cb;
    g.ldc = ldc;
    g.r = residual;
    g.ldr = ldr;
    return launch_tile(p.tile, 1, swiglu, g, stream);
  }
  g.c = part;
  g.ldc = (int)n4;
  g.slab = (size_t)m * n4;
  const hipError_t e = launch_tile(p.tile, p.splits, false, g, stream);
  if (e != hipSuccess) return e;
  const uintptr_t out = cb != nullptr ? (uintptr_t)cb : (uintptr_t)c;
  const int vec = n % 4 == 0 && ldc % 4 == 0 && (out & 15u) == 0;
  const unsigned bx = (n4 / 4 + 63) / 64;
  const unsigned by = std::min<unsigned>((m + 3) / 4, std::max(1u, 4096u / bx));
  hipLaunchKernelGGL(bf16_splitk_reduce_kernel, dim3(bx, by), dim3(256), 0, stream, part, g.slab, p.splits, (int)n4, c,
                     cb, ldc, residual, ldr, (int)m, (int)n, vec);
  return hipGetLastError();
}

namespace {

// dst [rows][ld_d] = src [rows][cols] (row pitch ld_s, any 2-byte alignment), zero
// from column cols on: eight values per thread, read with one unaligned 16-byte
// load, written with one store.
__global__ __launch_bounds__(256) void pad_rows16_kernel(const uint16_t* __restrict__ src, uint16_t* __restrict__ dst,
                                                         int rows, int cols, int ld_s, int ld_d) {
  const int c = (int)(blockIdx.x * 64 + (threadIdx.x & 63)) * 8;
  if (c >= ld_d) return;
  for (int r = (int)(blockIdx.y * 4 + (threadIdx.x >> 6)); r < rows; r += (int)gridDim.y * 4) {
    const uint16_t* p = src + (size_t)r * ld_s + c;
    uint16_t v[8];
    if (c + 8 <= cols) {
      __builtin_memcpy(v, p, 16);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = c + j < cols ? p[j] : (uint16_t)0;
    }
    __builtin_memcpy(__builtin_assume_aligned(dst + (size_t)r * ld_d + c, 16), v, 16);
  }
}

}  // namespace

hipError_t launch_bf16_pad_rows(const uint16_t* src, uint16_t* dst, uint32_t rows, uint32_t cols, int ld_s, int ld_d,
                                hipStream_t stream) {
  const unsigned bx = (unsigned)((ld_d / 8 + 63) / 64);
  const unsigned by = std::min<unsigned>((rows + 3) / 4, std::max(1u, 8192u / bx));
  hipLaunchKernelGGL(pad_rows16_kernel, dim3(bx, by), dim3(256), 0, stream, src, dst, (int)rows, (int)cols, ld_s,
                     ld_d);
  return hipGetLastError();
}

}  // namespace prom
