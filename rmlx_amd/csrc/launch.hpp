// Kernel launches with plain arguments.  Those are in scalar registers when a wave starts (-amdgpu-kernarg-preload-count; up to about 14
// dwords), a struct passed by value is loaded from memory first; but the runtime copies arguments one by one and looks up the allocation behind
// every one that is declared a pointer, 0.1 to 0.3 us a launch, and it looks the kernel up by its host address (0.16 us).  Here the handle is
// looked up once per kernel and device, the arguments are packed as the device reads them, and pointers travel as numbers.  A call of a small
// matmul, host bound: 3.25 to 3.4 us with a struct, 3.5 with plain arguments, 3.15 to 3.3 so.
#pragma once
#include <atomic>
#include <cstring>

#include "common.hpp"

namespace rmlx {

// A device pointer on its way through a plain argument, and in the kernel again: to global memory, as the compiler knows it of pointer arguments.
inline uint64_t address(const void* p) { return reinterpret_cast<uint64_t>(p); }
template <typename T>
__device__ __forceinline__ const T* global_at(uint64_t a) {
  return (const T*)(const __attribute__((address_space(1))) T*)a;
}

// The error of this thread's launches since it was last asked for (each launch's own result: asking the runtime for its last error would cost
// another 50 ns).
inline hipError_t& launch_error() {
  thread_local hipError_t e = hipSuccess;
  return e;
}
inline hipError_t take_launch_error() {
  const hipError_t e = launch_error();
  launch_error() = hipSuccess;
  if (e != hipSuccess) (void)hipGetLastError();  // (the runtime keeps it too, and other launches ask the runtime)
  return e;
}

template <auto Kernel>
struct Launch;
template <typename... P, void (*Kernel)(P...)>
struct Launch<Kernel> {
  static void go(dim3 grid, dim3 block, size_t lds, hipStream_t s, const P&... args) {
    constexpr int kDevices = 16;
    static std::atomic<hipFunction_t> known[kDevices];
    const int device = ctx().device;
    hipFunction_t f = device >= 0 && device < kDevices ? known[device].load(std::memory_order_relaxed) : nullptr;
    if (f == nullptr) {  // (of the current device, which is the library's in every entry point; two threads that look it up find the same)
      const hipError_t e = hipGetFuncBySymbol(&f, reinterpret_cast<const void*>(Kernel));
      if (e != hipSuccess) { launch_error() = e; return; }
      if (device >= 0 && device < kDevices) known[device].store(f, std::memory_order_relaxed);
    }
    alignas(16) char packed[(sizeof(P) + ... + 0) + 16 * sizeof...(P)];
    size_t at = 0;
    auto put = [&](const auto& v) {
      at = (at + alignof(decltype(v)) - 1) / alignof(decltype(v)) * alignof(decltype(v));
      std::memcpy(packed + at, &v, sizeof(v));
      at += sizeof(v);
    };
    (put(args), ...);
    void* extra[] = {HIP_LAUNCH_PARAM_BUFFER_POINTER, packed, HIP_LAUNCH_PARAM_BUFFER_SIZE, &at, HIP_LAUNCH_PARAM_END};
    const hipError_t e = hipModuleLaunchKernel(f, grid.x, grid.y, grid.z, block.x, block.y, block.z, (unsigned)lds, s, nullptr, extra);
    if (e != hipSuccess) launch_error() = e;
  }
};

}  // namespace rmlx
