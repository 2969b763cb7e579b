// The launches of oct_amd/csrc/reduction.hip, recorded instead of run: the HIP calls
// are defined here.  argv: rows width.  Fails (status 1) where the RMSNorm of a rows x
// width input is refused, a launch has 2^32 threads or more, which HIP refuses, or the
// launches do not take the rows one after the other, each once.
#include <stdio.h>
#include <stdlib.h>

#include <map>
#include <string>

#include "../oct_amd/csrc/reactor_internal.h"

namespace {
std::map<const void*, std::string> g_kernels;
dim3 g_grid, g_block;
const char* const kIn = reinterpret_cast<const char*>(1ull << 40);
char* const kOut = reinterpret_cast<char*>(1ull << 42);
char* const kInv = reinterpret_cast<char*>(1ull << 44);
uint64_t g_next_row = 0, g_width = 0;
bool g_wrong = false;
}  // namespace

namespace prom {
DeviceContext& ctx() {
  static DeviceContext context;
  return context;
}
void* staging(uint32_t, size_t) { return reinterpret_cast<void*>(1ull << 45); }
}  // namespace prom

extern "C" {
hipError_t hipGetLastError(void) { return hipSuccess; }
// row_kernel(in, w, out, aux, rows, width, stride, eps)
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t, hipStream_t) {
  if (g_kernels[f].find("row_kernel") == std::string::npos) return hipErrorInvalidDeviceFunction;
  const uint64_t threads = (uint64_t)grid.x * block.x;
  const uint32_t rows = *static_cast<uint32_t*>(args[4]);
  printf("row %llu: %u rows, %llu threads\n", (unsigned long long)g_next_row, rows, (unsigned long long)threads);
  if (threads >= 1ull << 32) g_wrong = true;
  if (*static_cast<const char**>(args[0]) != kIn + 4 * g_next_row * g_width) g_wrong = true;
  if (*static_cast<char**>(args[2]) != kOut + 4 * g_next_row * g_width) g_wrong = true;
  if (*static_cast<char**>(args[3]) != kInv + 4 * g_next_row) g_wrong = true;
  if (threads / 64 < rows) g_wrong = true;  // a wave per row at least
  g_next_row += rows;
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

int main(int argc, char** argv) {
  if (argc < 3) return 2;
  const uint32_t rows = (uint32_t)strtoul(argv[1], nullptr, 10), width = (uint32_t)strtoul(argv[2], nullptr, 10);
  g_width = width;
  const hipError_t e = prom::launch_rmsnorm(
      reinterpret_cast<const float*>(kIn), reinterpret_cast<const float*>(kIn), reinterpret_cast<float*>(kOut),
      reinterpret_cast<float*>(kInv), rows, width, width, 1e-6f, nullptr);
  return e != hipSuccess || g_wrong || g_next_row != rows;
}
