// A kernel's launch from the library's host code.
//
// A short call is host time, and most of that is the runtime's own launch.  Three things in a caller's hands move it (us
// of host time a launch of an empty kernel, back to back, on an MI355X's host):
//   - pointers as arguments.  The runtime looks every one of them up among its allocations: six pointers and four
//     scalars 3.6 to 4.1, the same bytes as one struct 2.65, as words 2.8.  So a kernel takes one struct.
//   - the argument record.  Up to 112 bytes a launch takes 2.75, from 116 on 3.6 (the record is written out to the
//     device).  A kernel that asks for its grid or workgroup size gets 256 bytes of hidden arguments behind its own: the
//     kernels here take what they need of those as an argument.
//   - the way in.  hipLaunchKernel looks the host symbol up on every call; a function handle, looked up once a device,
//     saves 0.12.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

namespace svodk {

template <auto Kernel>
struct Launch;

template <typename... P, void (*Kernel)(P...)>
struct Launch<Kernel> {
  // `lds`: dynamic LDS of this launch, `most_lds`: the most any launch of the kernel asks for.
  // The current device is the stream's (the op layer sees to it): the function looked up is that device's.
  static hipError_t run(int64_t grid, uint32_t block, uint32_t lds, uint32_t most_lds, hipStream_t stream, P... args) {
    constexpr int kDevices = 16;  // devices past these look the function up every time
    static std::atomic<hipFunction_t> known[kDevices];
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    hipFunction_t f = device >= 0 && device < kDevices ? known[device].load(std::memory_order_acquire) : nullptr;
    if (f == nullptr) {
      // Two threads that both get here ask the runtime twice and store the same answer.
      if (most_lds > 64 * 1024) {
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(Kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)most_lds);
        if (e != hipSuccess) return e;
      }
      e = hipGetFuncBySymbol(&f, reinterpret_cast<const void *>(Kernel));
      if (e != hipSuccess) return e;
      if (device >= 0 && device < kDevices) known[device].store(f, std::memory_order_release);
    }
    void *at[] = {&args...};
    return hipModuleLaunchKernel(f, (uint32_t)grid, 1, 1, block, 1, 1, lds, stream, at, nullptr);
  }
};

}  // namespace svodk
