// Kernel launches recorded instead of run, for checks of host code linked without the HIP
// runtime: each goes to recorded_launch(kernel's mangled name, grid, block, arguments).
// No device: the runtime's context is empty, staging buffers are addresses that nobody reads.
#pragma once
#include <map>
#include <string>

#include "../oct_amd/csrc/reactor_internal.h"

hipError_t recorded_launch(const std::string& kernel, dim3 grid, dim3 block, void** args);

namespace {
std::map<const void*, std::string> g_kernels;
dim3 g_grid, g_block;
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
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t, hipStream_t) {
  return recorded_launch(g_kernels[f], grid, block, args);
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
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
}
