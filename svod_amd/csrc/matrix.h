// What the two kernels of linear share: the matrix instruction, the buffer descriptor of a fill, four elements at a time.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "convert.h"

namespace svodk {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
typedef __attribute__((ext_vector_type(4))) int i32x4;

template <bool F16>
__device__ __forceinline__ f32x4 mma(const u32x4 &a, const u32x4 &b, const f32x4 &c) {
#if defined(__HIP_DEVICE_COMPILE__)
  if constexpr (F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
#else
  return c;
#endif
}

// Past every descriptor's bound: a lane that fetches from there lands zeros.
constexpr uint32_t kPastBound = 0xfffffff0u;

// A raw buffer descriptor over `bytes` bytes at `base`: loads past the end return zero.
__device__ __forceinline__ i32x4 make_rsrc(const void *base, int64_t bytes) {
  const int64_t clamped = bytes < 0 ? 0 : (bytes > (int64_t)kPastBound ? (int64_t)kPastBound : bytes);
  const uint64_t addr = (uint64_t)(uintptr_t)base;
  return i32x4{(int)(uint32_t)addr, (int)(uint32_t)((addr >> 32) & 0xffffu), (int)(uint32_t)clamped, 0x00020000};
}

// Four 16-bit elements at `p` (8-byte aligned) as f32.
template <bool F16>
__device__ __forceinline__ f32x4 load4(const uint16_t *p) {
  const u32x2 x = *reinterpret_cast<const u32x2 *>(p);
  if constexpr (F16) {
    const f32x2 lo = __builtin_convertvector(__builtin_bit_cast(f16x2, (uint32_t)x[0]), f32x2);
    const f32x2 hi = __builtin_convertvector(__builtin_bit_cast(f16x2, (uint32_t)x[1]), f32x2);
    return f32x4{lo[0], lo[1], hi[0], hi[1]};
  } else {
    return f32x4{bf16_lo(x[0]), bf16_hi(x[0]), bf16_lo(x[1]), bf16_hi(x[1])};
  }
}

}  // namespace svodk
