// Matrix products of 16-bit operands, LDS-DMA and its waits, shared by the kernels of this directory.
#pragma once
#include "seqmix.h"

namespace lumen {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// 16 x 16 x 32
template <typename T> struct Mfma;
template <> struct Mfma<bf16> {
  static __device__ __forceinline__ f32x4 run(uint4 a, uint4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <> struct Mfma<fp16> {
  static __device__ __forceinline__ f32x4 run(uint4 a, uint4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};

// 32 x 32 x 16
template <typename T> struct Mma32;
template <> struct Mma32<bf16> {
  static __device__ __forceinline__ f32x16 run(uint4 a, uint4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <> struct Mma32<fp16> {
  static __device__ __forceinline__ f32x16 run(uint4 a, uint4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};

// the two halves of a packed 16-bit pair as fp32 (bf16: a shift and a mask)
template <typename T> __device__ __forceinline__ void unpack2(unsigned v, float& a, float& b);
template <> __device__ __forceinline__ void unpack2<bf16>(unsigned v, float& a, float& b) {
  a = __uint_as_float(v << 16);
  b = __uint_as_float(v & 0xffff0000u);
}
template <> __device__ __forceinline__ void unpack2<fp16>(unsigned v, float& a, float& b) {
  const lumen_f16x2 h = __builtin_bit_cast(lumen_f16x2, v);
  a = static_cast<float>(h[0]);
  b = static_cast<float>(h[1]);
}

// prompt attention: log of the largest weight a tile may form before its maximum moves the reference
constexpr float kRise = 5.f;

// at most N vector loads are left in flight
template <int N> __device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0xF70);
}

// LDS-DMA of 16 bytes per lane (wave-uniform base, 32-bit lane offset, LDS address of the wave's 1-KiB piece).  Inline
// asm, so that a kernel's own counted waits order it.
__device__ __forceinline__ void dma16(const void* base, unsigned off, unsigned lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :: "v"(off), "s"(base), "s"(lds) : "memory", "m0");
}

}  // namespace lumen
