// Prints the kernel that the GeGLU product of argv (rows, columns of each half, k) runs on:
// "rows", "tiles", or "none" where it is not fused.  The launches are recorded, not run.
#include <stdio.h>
#include <stdlib.h>

#include "recorded_launches.h"

hipError_t recorded_launch(const std::string& kernel, dim3, dim3, void**) {
  puts(kernel.find("sgemm_rows_kernel") != std::string::npos ? "rows"
       : kernel.find("geglu") != std::string::npos           ? "tiles"
                                                              : kernel.c_str());
  return hipSuccess;
}
extern "C" hipError_t hipGetSymbolAddress(void**, const void*) { return hipErrorInvalidSymbol; }

int main(int argc, char** argv) {
  if (argc < 4) return 2;
  const uint32_t m = (uint32_t)atoi(argv[1]), f = (uint32_t)atoi(argv[2]), k = (uint32_t)atoi(argv[3]);
  float* const at = reinterpret_cast<float*>(1ull << 40);
  const hipError_t e = prom::launch_sgemm_f32_geglu(at, (int)k, at, at, (int)f, m, f, k, nullptr);
  if (e == hipErrorNotSupported) puts("none");
  return e != hipSuccess && e != hipErrorNotSupported;
}
