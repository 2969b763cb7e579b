// The launches of oct_amd/csrc/reduction.hip, recorded instead of run.  argv: rows width.
// Fails (status 1) where the RMSNorm of a rows x width input is refused, a launch has
// 2^32 threads or more, which HIP refuses, or the launches do not take the rows one
// after the other, each once.
#include <stdio.h>
#include <stdlib.h>

#include "recorded_launches.h"

namespace {
const char* const kIn = reinterpret_cast<const char*>(1ull << 40);
char* const kOut = reinterpret_cast<char*>(1ull << 42);
char* const kInv = reinterpret_cast<char*>(1ull << 44);
uint64_t g_next_row = 0, g_width = 0;
bool g_wrong = false;
}  // namespace

// row_kernel(in, w, out, aux, rows, width, stride, eps)
hipError_t recorded_launch(const std::string& kernel, dim3 grid, dim3 block, void** args) {
  if (kernel.find("row_kernel") == std::string::npos) return hipErrorInvalidDeviceFunction;
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

int main(int argc, char** argv) {
  if (argc < 3) return 2;
  const uint32_t rows = (uint32_t)strtoul(argv[1], nullptr, 10), width = (uint32_t)strtoul(argv[2], nullptr, 10);
  g_width = width;
  const hipError_t e = prom::launch_rmsnorm(
      reinterpret_cast<const float*>(kIn), reinterpret_cast<const float*>(kIn), reinterpret_cast<float*>(kOut),
      reinterpret_cast<float*>(kInv), rows, width, width, 1e-6f, nullptr);
  return e != hipSuccess || g_wrong || g_next_row != rows;
}
