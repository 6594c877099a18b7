// Prints the plan of GEMM calls (plan_gemm, csrc/gemm.hip) on the host: which
// kernel and which instance a call takes, and the scratch it needs. Reads lines
//   <f16|f32> M N K A-offset B-offset capacity
// (offsets in elements from an aligned address; capacity in bytes, 0: a *_ws
// call's) and answers each with "key=value" words. gemm.hip is compiled for the
// host only; no kernel can be launched, and the HIP calls that a plan makes are
// answered here, for a GPU of 256 CUs. The addresses are never read.

#include <cstdio>

#include "gemm.hip"

extern "C" {
hipError_t hipGetDevice(int* device) {
  *device = 0;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* value, hipDeviceAttribute_t, int) {
  *value = 256;
  return hipSuccess;
}
// The registration of the device code that a host-only object does not have.
char __hip_fatbin;
void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*,
                           void*, int*) {}
void __hipUnregisterFatBinary(void**) {}
}

namespace {

template <typename T>
void answer(int m, int n, int k, int a_off, int b_off, std::size_t capacity) {
  const T* const a = reinterpret_cast<const T*>(std::uintptr_t(1) << 40) + a_off;
  const T* const b = reinterpret_cast<const T*>(std::uintptr_t(2) << 40) + b_off;
  const GemmPlan p = plan_gemm<T>(a, b, m, n, k, capacity > 0 ? capacity : opl::kUnlimited);
  const char* const kinds[] = {"skinny", "narrow", "split", "dma", "register"};
  std::printf("kind=%s bytes=%zu", kinds[p.kind], p.bytes);
  if (p.kind == GemmPlan::kSkinny)
    std::printf(" splits=%d mfma=%d", p.skinny.splits, m >= skinny::Cfg<T>::kMfmaMinM);
  if (p.kind == GemmPlan::kSplit) {
    const int step = (p.split.deep && sizeof(T) == 2 && p.split.fm > 1 ? 2 : 1) *
                     dma::Elem<T>::kSubK;
    std::printf(" fm=%d splits=%d deep=%d edge=%d", p.split.fm, p.split.splits,
                step > dma::Elem<T>::kSubK, k % step != 0 || (sizeof(T) == 2 && n % 2 != 0));
  }
  if (p.kind == GemmPlan::kDma) {
    const bool small = (m + 255LL) / 256 * ((n + 255LL) / 256) < DmaTiles<T>::kSmallBelow;
    const int one_round = DmaTiles<T>::kOneRound ? one_round_rows(m, n) : 0;
    std::printf(" rows=%d tail=%d pad=%d", one_round > 0 ? one_round : small ? 128 : 256,
                p.tail.splits, p.pad.pad_a + 2 * p.pad.pad_b);
    if (one_round > 0) std::printf(" one_round=1");
  }
  if (p.kind == GemmPlan::kRegister) std::printf(" staging=%d", p.staging);
  std::puts("");
}

}  // namespace

int main() {
  char type[8];
  int m, n, k, a_off, b_off;
  std::size_t capacity;
  while (std::scanf("%7s %d %d %d %d %d %zu", type, &m, &n, &k, &a_off, &b_off, &capacity) == 7) {
    if (type[1] == '1')
      answer<_Float16>(m, n, k, a_off, b_off, capacity);
    else
      answer<float>(m, n, k, a_off, b_off, capacity);
  }
  return 0;
}
