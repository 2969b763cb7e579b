// Host <-> device copies of caller-owned (pageable) host buffers.
//
// The host-pointer entry points (prometheus_reactor_runtime_sgemm and the
// other calls that take host arrays, reactor_sgemm.cpp:4152-4191) receive
// ordinary pageable memory.  HIP copies such memory through its own staging
// at 8-23 GB/s host-to-device and ~17 GB/s device-to-host on MI355X, while
// DMA from pinned memory runs at ~57 GB/s both ways, and a small pageable copy
// costs 10-40 us of calls (two 64 KiB uploads, a kernel and a download: 102 us;
// through pinned memory 22).  So every copy goes through pinned memory:
//   * up to 512 KiB in one piece, moved by a copy kernel on the compute queue,
//     which reads or writes the pinned memory itself: at these sizes a DMA copy
//     spends more time handing over between the copy engine and the queue than
//     copying (3 copies of 64 KiB and a kernel: 38 us by DMA, 22 by kernels);
//   * larger ones in chunks of half the copy, 1 to 8 MiB: the host threads copy
//     chunk i into a pinned slot while chunk i-1 moves, and the reverse for
//     downloads (a slot is written again only when an event behind every copy from it
//     has passed: Ring).  Four host threads (the caller and three workers) copy pageable
//     <-> pinned at 70-95 GB/s (one: 30); the pipelined upload of 64 MiB measured 47
//     GB/s.  Two chunks keep a copy of a few MiB, which was one, from running host
//     and device in turn; below 4 MiB they move by the copy kernel too, since each
//     DMA copy adds ~15 us (three copies of 4 MiB in chunks of 4, 2, 1, 0.5 MiB: by
//     DMA 365, 348, 394, 523 us, by kernels 368, 315, 323, 480).
// The host-pointer SGEMM, us before and after: 32^3 34 -> 24, 256^3 71 -> 57, 512^3
// 164 -> 127, 1024^3 470 -> 380, 1536^3 932 -> 835.
// Without pinned memory the copies keep hipMemcpyAsync.  host_memcpy lends the
// same threads to the async and batch entries' copies between caller buffers and
// their own pinned staging.  Nothing here changes what is copied, only how.
#include <string.h>

#include <atomic>
#include <condition_variable>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>

#include "reactor_internal.h"

namespace prom {
namespace {

constexpr size_t kLargeSlot = 8u << 20;  // slots of the chunked copies, and their largest chunk
constexpr size_t kSmallSlot = 1u << 20;  // slots of the copies made in one piece
constexpr size_t kSmallMax = 512u << 10;
constexpr size_t kChunkMin = 1u << 20;
constexpr size_t kKernelMax = 4u << 20;  // pieces below this move by the copy kernel
constexpr int kSlots = 4;
constexpr int kCopyThreads = 4;
constexpr size_t kParallelMin = 768u << 10;

// One or two pieces copied by the calling thread and up to kCopyThreads - 1
// persistent workers.  The threads claim blocks (an eighth of a piece, 256 KiB or
// more) in order, so the
// caller never waits for a worker that has not been scheduled yet (waking idle cores
// takes up to ~100 us, and milliseconds on busy ones): it copies what nobody has
// claimed and waits only for blocks that are being copied.  One job at a time
// (callers hold the pipe's mutex).  The workers are never joined: they wait on the
// condition variable until the process ends, and the pool is never destroyed, so no
// exit-time destructor races them.
class CopyPool {
 public:
  struct Piece {
    char* dst;
    const char* src;
    size_t bytes;
  };

  void begin(const Piece* pieces, int n) {
    uint64_t blocks = 0;
    block_ = std::max<size_t>(256u << 10, (pieces[0].bytes / 8 + 65535) & ~(size_t)65535);
    for (int c = 0; c < 2; ++c) {
      piece_[c] = c < n ? pieces[c] : Piece{nullptr, nullptr, 0};
      first_[c] = blocks;
      blocks += (piece_[c].bytes + block_ - 1) / block_;
      done_[c].store(0, std::memory_order_relaxed);
    }
    first_[2] = blocks;
    const bool shared = piece_[0].bytes + piece_[1].bytes >= kParallelMin && start();
    {
      std::lock_guard<std::mutex> g(mu_);
      ++generation_;
      claim_.store(pack(generation_, blocks, 0), std::memory_order_release);
    }
    if (shared) work_.notify_all();
  }
  // Returns when piece c is copied.
  void finish(int c) {
    const uint64_t mine = first_[c + 1] - first_[c];
    while (done_[c].load(std::memory_order_acquire) < mine)
      if (!copy_block(generation_, first_[c + 1])) std::this_thread::yield();
  }
  void copy(char* dst, const char* src, size_t bytes) {
    const Piece one{dst, src, bytes};
    begin(&one, 1);
    finish(0);
  }

 private:
  // generation (24 bits) | blocks (20) | next block (20): a thread claims a block of
  // the generation it knows with one exchange, so a late worker never takes another
  // job's block, and a job's fields do not change while a block of it is claimed.
  static uint64_t pack(uint64_t gen, uint64_t blocks, uint64_t next) {
    return (gen & 0xffffffu) << 40 | blocks << 20 | next;
  }
  bool copy_block(uint64_t gen, uint64_t below) {
    uint64_t v = claim_.load(std::memory_order_acquire), next;
    do {
      next = v & 0xfffffu;
      if (v >> 40 != (gen & 0xffffffu) || next >= ((v >> 20) & 0xfffffu) || next >= below) return false;
    } while (!claim_.compare_exchange_weak(v, v + 1, std::memory_order_acq_rel, std::memory_order_acquire));
    const int c = next >= first_[1];
    const Piece& p = piece_[c];
    const size_t off = (size_t)(next - first_[c]) * block_;
    memcpy(p.dst + off, p.src + off, std::min(block_, p.bytes - off));
    done_[c].fetch_add(1, std::memory_order_release);
    return true;
  }
  bool start() {
    if (started_) return threads_ > 1;
    started_ = true;
    std::lock_guard<std::mutex> g(mu_);
    for (int id = 1; id < kCopyThreads; ++id) {
      try {
        std::thread([this] { worker(); }).detach();
        threads_ = id + 1;
      } catch (const std::system_error&) {
        break;
      }
    }
    return threads_ > 1;
  }
  void worker() {
    uint64_t seen = 0;
    for (;;) {
      {
        std::unique_lock<std::mutex> g(mu_);
        work_.wait(g, [&] { return generation_ != seen; });
        seen = generation_;
      }
      while (copy_block(seen, ~0ull)) {
      }
    }
  }

  std::mutex mu_;
  std::condition_variable work_;
  bool started_ = false;
  int threads_ = 1;
  uint64_t generation_ = 0;  // written under mu_ by the caller of the job
  size_t block_ = 0;
  Piece piece_[2] = {};
  uint64_t first_[3] = {};  // first block of each piece, and the end
  std::atomic<uint64_t> claim_{0}, done_[2] = {};
};

// `bytes` from src to dst, one of them pinned host memory, both 16-byte aligned.
__global__ __launch_bounds__(256) void pinned_copy_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst,
                                                          size_t bytes) {
  const size_t n = bytes / 16;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) dst[i] = src[i];
  const size_t rest = bytes - 16 * n;
  if (blockIdx.x == 0 && threadIdx.x < rest)
    reinterpret_cast<char*>(dst + n)[threadIdx.x] = reinterpret_cast<const char*>(src + n)[threadIdx.x];
}

// A ring of kSlots pinned slots.  take() hands out consecutive regions of the
// current slot; a slot is left with an event behind its last copy and entered
// again only once that event has passed.  The event covers what is queued when
// take() leaves the slot, so the copies of every region taken before have to be
// queued by then: pieces that are filled together are parts of one region.
struct Ring {
  size_t slot_bytes = 0;
  bool tried = false, ready = false;
  char* slot[kSlots] = {};
  hipEvent_t done[kSlots] = {};
  bool busy[kSlots] = {};  // done[i] was recorded and not yet waited for
  int current = 0;
  size_t used = 0;
  hipStream_t stream = nullptr;  // of the copies in the current slot

  // The slots and events, made at the first use and kept for the process.
  bool init(size_t bytes) {
    if (tried) return ready;
    tried = true;
    slot_bytes = bytes;
    for (int i = 0; i < kSlots; ++i) {
      // Coherent: the copy kernel must see what the host wrote since its last launch.
      if (hipHostMalloc(reinterpret_cast<void**>(&slot[i]), bytes, hipHostMallocCoherent) != hipSuccess ||
          hipEventCreateWithFlags(&done[i], hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();
        return false;
      }
    }
    ready = true;
    return true;
  }
  // `bytes` <= slot_bytes for copies on st; null: *e says why, and the ring stays in
  // its slot.
  char* take(size_t bytes, hipStream_t st, hipError_t* e) {
    *e = hipSuccess;
    if (used > 0 && (st != stream || used + bytes > slot_bytes)) {
      *e = hipEventRecord(done[current], stream);
      if (*e != hipSuccess) return nullptr;
      busy[current] = true;
      const int next = (current + 1) % kSlots;
      if (busy[next]) {
        *e = hipEventSynchronize(done[next]);
        if (*e != hipSuccess) return nullptr;
        busy[next] = false;
      }
      current = next;
      used = 0;
    }
    stream = st;
    char* p = slot[current] + used;
    used += (bytes + 255) & ~(size_t)255;
    return p;
  }
};

struct Pipe {
  std::mutex mu;
  Ring small, large;
  hipEvent_t chunk_done[kSlots] = {};  // downloads: chunk i is in its slot
  bool chunk_events = false;
  CopyPool pool;

  // The ring for a copy of `bytes` and the size of its pieces; null without pinned memory.
  Ring* ring(size_t bytes, size_t* piece) {
    if (bytes <= kSmallMax) {
      *piece = bytes;
      return small.init(kSmallSlot) ? &small : nullptr;
    }
    if (!large.init(kLargeSlot)) return nullptr;
    if (!chunk_events) {
      for (hipEvent_t& ev : chunk_done)
        if (hipEventCreateWithFlags(&ev, hipEventDisableTiming) != hipSuccess) {
          (void)hipGetLastError();
          return nullptr;
        }
      chunk_events = true;
    }
    const size_t half = (bytes / 2 + 65535) & ~(size_t)65535;
    *piece = std::min(kLargeSlot, std::max(kChunkMin, half));
    return &large;
  }
};

// One piece between pinned and device memory.
hipError_t move(void* dst, const void* src, size_t bytes, hipMemcpyKind kind, hipStream_t stream) {
  if (bytes >= kKernelMax || ((reinterpret_cast<uintptr_t>(dst) | reinterpret_cast<uintptr_t>(src)) & 15) != 0)
    return hipMemcpyAsync(dst, src, bytes, kind, stream);
  const unsigned blocks = (unsigned)std::min<size_t>(64, (bytes + 4095) / 4096);
  hipLaunchKernelGGL(pinned_copy_kernel, dim3(blocks), dim3(256), 0, stream, static_cast<const uint4*>(src),
                     static_cast<uint4*>(dst), bytes);
  return hipGetLastError();
}

Pipe& pipe() {
  static Pipe* p = new Pipe();  // never destroyed (its workers outlive static destruction)
  return *p;
}

}  // namespace

void host_memcpy(void* dst, const void* src, size_t bytes) {
  if (bytes < kParallelMin) {
    memcpy(dst, src, bytes);
    return;
  }
  Pipe& p = pipe();
  std::lock_guard<std::mutex> g(p.mu);
  p.pool.copy(static_cast<char*>(dst), static_cast<const char*>(src), bytes);
}

hipError_t upload_host(void* dst, const void* src, size_t bytes, hipStream_t stream) {
  if (bytes == 0) return hipSuccess;
  Pipe& p = pipe();
  std::lock_guard<std::mutex> g(p.mu);
  size_t piece = 0;
  Ring* ring = p.ring(bytes, &piece);
  if (ring == nullptr) return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, stream);
  const char* s8 = static_cast<const char*>(src);
  char* d8 = static_cast<char*>(dst);
  // A copy of two pieces below 4 MiB is one job in one region of a slot; larger ones go
  // piece by piece, so that no piece waits for a slot before its turn.
  const size_t region = bytes <= 2 * piece && piece < kKernelMax ? bytes : piece;
  for (size_t off = 0; off < bytes;) {
    const size_t all = std::min(region, bytes - off);
    hipError_t e;
    char* const pinned = ring->take(all, stream, &e);
    if (pinned == nullptr) return e;
    CopyPool::Piece job[2];
    int n = 0;
    for (size_t at = 0; at < all; at += piece, ++n)
      job[n] = {pinned + at, s8 + off + at, std::min(piece, all - at)};
    p.pool.begin(job, n);
    hipError_t first = hipSuccess;
    for (int c = 0; c < n; ++c) {
      p.pool.finish(c);  // also after an error: the job has to end
      if (first == hipSuccess) first = move(d8 + off, job[c].dst, job[c].bytes, hipMemcpyHostToDevice, stream);
      off += job[c].bytes;
    }
    if (first != hipSuccess) return first;
  }
  return hipSuccess;
}

hipError_t download_host(void* dst, const void* src, size_t bytes, hipStream_t stream) {
  if (bytes == 0) return hipSuccess;
  Pipe& p = pipe();
  std::lock_guard<std::mutex> g(p.mu);
  size_t piece = 0;
  Ring* ring = p.ring(bytes, &piece);
  if (ring == nullptr) {
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream);
    return e != hipSuccess ? e : hipStreamSynchronize(stream);
  }
  const char* s8 = static_cast<const char*>(src);
  char* d8 = static_cast<char*>(dst);
  if (bytes <= piece) {
    hipError_t e;
    char* pinned = ring->take(bytes, stream, &e);
    if (pinned == nullptr) return e;
    e = move(pinned, src, bytes, hipMemcpyDeviceToHost, stream);
    if (e == hipSuccess) e = hipStreamSynchronize(stream);
    if (e == hipSuccess) p.pool.copy(d8, pinned, bytes);
    return e;
  }
  // Up to kSlots pieces are queued ahead of the host copies; piece i is copied out
  // before piece i + kSlots is queued, so no piece's region is taken again early, and
  // each piece's move is queued before the next region is taken.
  const size_t chunks = (bytes + piece - 1) / piece;
  char* pinned[kSlots] = {};
  auto length = [&](size_t i) { return std::min(piece, bytes - i * piece); };
  auto enqueue = [&](size_t i) -> hipError_t {
    hipError_t e;
    char* at = ring->take(length(i), stream, &e);
    if (at == nullptr) return e;
    pinned[i % kSlots] = at;
    e = move(at, s8 + i * piece, length(i), hipMemcpyDeviceToHost, stream);
    return e != hipSuccess ? e : hipEventRecord(p.chunk_done[i % kSlots], stream);
  };
  for (size_t i = 0; i < chunks && i < (size_t)kSlots; ++i) {
    const hipError_t e = enqueue(i);
    if (e != hipSuccess) return e;
  }
  for (size_t i = 0; i < chunks; ++i) {
    hipError_t e = hipEventSynchronize(p.chunk_done[i % kSlots]);
    if (e != hipSuccess) return e;
    p.pool.copy(d8 + i * piece, pinned[i % kSlots], length(i));
    if (i + kSlots < chunks) {
      e = enqueue(i + kSlots);
      if (e != hipSuccess) return e;
    }
  }
  return hipSuccess;
}

}  // namespace prom
