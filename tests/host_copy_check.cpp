// The host copies (oct_amd/csrc/host_copy.hip) against a device that runs late: the HIP
// calls they make are defined here, every copy is queued, and the queue runs only as
// far as a wait asks for.  A pinned slot that is written again before its copy has
// been waited for therefore always shows as wrong data.
//
// argv[1]: "uploads" mixed sizes, one after the other without waits; "mixed" downloads
// among them; "errors" waits and copies that fail now and then.  Prints what differed; exit
// status 1 then.
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <functional>
#include <map>
#include <string>
#include <vector>

#include "../oct_amd/csrc/reactor_internal.h"

namespace {

std::vector<std::function<void()>> g_queue;
size_t g_run = 0;                        // operations that have run
std::map<hipEvent_t, size_t> g_events;   // operations before the event's record
std::map<const void*, std::string> g_kernels;
dim3 g_grid, g_block;
int g_fail_every = 0, g_fallible = 0;    // every so many waits and copies one fails

void run_to(size_t n) {
  for (; g_run < n; ++g_run) g_queue[g_run]();
}
bool fails() { return g_fail_every > 0 && ++g_fallible % g_fail_every == 0; }
void queue_copy(void* dst, const void* src, size_t bytes) {
  g_queue.push_back([=] { memcpy(dst, src, bytes); });
}

uint32_t g_random = 1;
uint32_t next_random() { return g_random = g_random * 1664525u + 1013904223u; }

}  // namespace

extern "C" {
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
  return posix_memalign(p, 4096, bytes) == 0 ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = reinterpret_cast<hipEvent_t>(new char);
  g_events[*e] = 0;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  g_events[e] = g_queue.size();
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  if (fails()) return hipErrorUnknown;
  run_to(g_events[e]);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  run_to(g_queue.size());
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind, hipStream_t) {
  if (fails()) return hipErrorUnknown;
  queue_copy(dst, src, bytes);
  return hipSuccess;
}
// The copy kernel is the only one: (const uint4* src, uint4* dst, size_t bytes).
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t) {
  if (g_kernels[f].find("pinned_copy_kernel") == std::string::npos) return hipErrorInvalidDeviceFunction;
  queue_copy(*static_cast<void**>(args[1]), *static_cast<void**>(args[0]), *static_cast<size_t*>(args[2]));
  return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t, hipStream_t) {
  g_grid = grid;
  g_block = block;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* stream) {
  *grid = g_grid;
  *block = g_block;
  *shared = 0;
  *stream = nullptr;
  return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) { return nullptr; }
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*,
                           int*) {
  g_kernels[f] = name;
}
void __hipUnregisterFatBinary(void**) {}
}

namespace {

struct Upload {
  std::vector<char> device;
  char value;
  bool ok;
};

size_t pick_bytes() {
  // the sizes of a product's operands: a few bytes to two and a half slots
  static const size_t kTop[] = {4096, 512u << 10, 1u << 20, 8u << 20, 20u << 20};
  return 1 + next_random() % kTop[next_random() % 5];
}

int check(const char* mode) {
  int wrong = 0;
  const bool downloads = strcmp(mode, "mixed") == 0, errors = strcmp(mode, "errors") == 0;
  if (errors) g_fail_every = 7;
  for (int round = 0; round < 40; ++round) {
    std::vector<Upload> all;
    for (int i = 0; i < 12; ++i) {
      // a short operand between two long ones first, then at random
      static const size_t kFirst[] = {5u << 20, 64u << 20, 5u << 20};
      const size_t bytes = round == 0 && i < 6 ? kFirst[i % 3] : pick_bytes();
      all.push_back(Upload{std::vector<char>(bytes, 0), (char)(1 + next_random() % 255), false});
      Upload& u = all.back();
      const std::vector<char> host(bytes, u.value);  // gone when the call returns
      u.ok = prom::upload_host(u.device.data(), host.data(), bytes, nullptr) == hipSuccess;
      if (!u.ok && !errors) {
        printf("round %d: upload %d of %zu bytes failed\n", round, i, bytes);
        return 1;
      }
      if (downloads && i % 3 == 2) {
        std::vector<char> back(all[i - 1].device.size(), 0);
        if (prom::download_host(back.data(), all[i - 1].device.data(), back.size(), nullptr) != hipSuccess) return 1;
        if (back != std::vector<char>(back.size(), all[i - 1].value)) {
          printf("round %d: download %d of %zu bytes differs\n", round, i, back.size());
          ++wrong;
        }
      }
    }
    (void)hipStreamSynchronize(nullptr);
    for (size_t i = 0; i < all.size(); ++i) {
      size_t bad = 0;
      for (const char c : all[i].device) bad += c != all[i].value;
      if (all[i].ok && bad > 0) {
        printf("round %d: upload %zu of %zu bytes: %zu differ\n", round, i, all[i].device.size(), bad);
        ++wrong;
      }
    }
    g_queue.clear();
    g_run = 0;
    for (auto& e : g_events) e.second = 0;  // all have passed
  }
  return wrong > 0;
}

}  // namespace

int main(int argc, char** argv) {
  const int status = check(argc > 1 ? argv[1] : "uploads");
  fflush(stdout);
  _Exit(status);  // the copy threads wait for work for ever
}
