// Prints the kernels that calls of the C ABI launch, on the host: the library's
// sources are compiled for the host only, and the HIP calls that a launch makes are
// answered here (for a GPU of 256 CUs), so nothing runs and the addresses are never
// read. Reads lines
//   <softmax|rmsnorm> <f16|f32> rows cols input-offset output-offset
//   attention <f16|f32> batch heads sequence head-dim causal
// (offsets in elements from an aligned address; softmax and RMSNorm through their
// workspace forms, which need no arena) and answers each with "status" and, for each
// launch, the kernel's mangled name and its grid.

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <cstring>
#include <map>
#include <string>

#include "operatorlib/operatorlib_c.h"

namespace {

// Host-side handle of a kernel -> its device name, as registered at start-up.
std::map<const void*, std::string>& kernels() {
  static std::map<const void*, std::string> names;
  return names;
}

dim3 pushed_grid, pushed_block;
std::string launched;

hipError_t record(const void* kernel, dim3 grid) {
  char text[64];
  std::snprintf(text, sizeof text, ":%ux%u", grid.x, grid.y);
  launched += " " + kernels()[kernel] + text;
  return hipSuccess;
}

}  // namespace

extern "C" {
char __hip_fatbin;
void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*,
                           void*, void*, void*, int*) {
  kernels()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t, hipStream_t) {
  pushed_grid = grid;
  pushed_block = block;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* stream) {
  *grid = pushed_grid;
  *block = pushed_block;
  *shared = 0;
  *stream = nullptr;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* kernel, dim3 grid, dim3, void**, size_t, hipStream_t) {
  return record(kernel, grid);
}
hipError_t hipExtLaunchKernel(const void* kernel, dim3 grid, dim3, void**, size_t, hipStream_t,
                              hipEvent_t, hipEvent_t, int) {
  return record(kernel, grid);
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetDevice(int* device) {
  *device = 0;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* value, hipDeviceAttribute_t, int) {
  *value = 256;
  return hipSuccess;
}
}

int main() {
  // aligned addresses, far apart
  auto f32 = [](int i, int offset = 0) {
    return reinterpret_cast<float*>(std::uintptr_t(i) << 40) + offset;
  };
  auto f16 = [](int i, int offset = 0) {
    return reinterpret_cast<operatorlib_half_t*>(std::uintptr_t(i) << 40) + offset;
  };
  void* const workspace = f32(9);
  const size_t bytes = size_t(1) << 30;
  char op[16], type[8];
  while (std::scanf("%15s %7s", op, type) == 2) {
    const bool half = type[1] == '1';
    launched.clear();
    int status = -1;
    if (std::strcmp(op, "attention") == 0) {
      int b, h, s, d, c;
      if (std::scanf("%d %d %d %d %d", &b, &h, &s, &d, &c) != 5) return 1;
      status = half ? operatorlib_attention_f16(f16(1), f16(2), f16(3), f32(4), b, h, s, d, c,
                                                nullptr)
                    : operatorlib_attention_f32(f32(1), f32(2), f32(3), f32(4), b, h, s, d, c,
                                                nullptr);
    } else {
      int rows, cols, in, out;
      if (std::scanf("%d %d %d %d", &rows, &cols, &in, &out) != 4) return 1;
      if (std::strcmp(op, "softmax") == 0)
        status = half ? operatorlib_softmax_f16_ws(f16(1, in), f16(2, out), rows, cols, workspace,
                                                   bytes, nullptr)
                      : operatorlib_softmax_f32_ws(f32(1, in), f32(2, out), rows, cols, workspace,
                                                   bytes, nullptr);
      else
        status = half ? operatorlib_rmsnorm_f16_ws(f16(1, in), f16(3), f16(2, out), rows, cols,
                                                   1e-6f, workspace, bytes, nullptr)
                      : operatorlib_rmsnorm_f32_ws(f32(1, in), f32(3), f32(2, out), rows, cols,
                                                   1e-6f, workspace, bytes, nullptr);
    }
    std::printf("%d%s\n", status, launched.c_str());
  }
  return 0;
}
