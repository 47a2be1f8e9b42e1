// The three codebooks, shared by the encoder and the storage kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <stdint.h>

typedef _Float16 f16;
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f16 f16_bits(uint32_t b) {
  return __builtin_bit_cast(f16, (uint16_t)b);
}
__device__ __forceinline__ uint16_t bits_f16(f16 h) { return __builtin_bit_cast(uint16_t, h); }

// The codebooks (reference trellis_format.py:41-81, quantize_kernels.sycl:51-73;
// upstream codebook.cuh:56-123) hash state s to x = s * M (+ A for 3INST)
// modulo 2^32 and decode x. The hash is affine in s, so for s = s1 + s2
// (disjoint bit fields) x = hash(s1) + s2 * M: the traceback trees compute
// one product per lane and add compile-time offsets for the other fields,
// instead of a quarter-rate v_mul_lo_u32 per leaf.
__host__ __device__ constexpr uint32_t hash_mult(int cb) {
  return cb == 2 ? 0x83DCD12Du : (cb == 0 ? 89226354u : 0xCBAC1FEDu);
}
__device__ __forceinline__ uint32_t hash_state(int cb, uint32_t s) {
  return s * hash_mult(cb) + (cb == 0 ? 64248484u : 0u);
}
__device__ __forceinline__ f16 decode_hash(int cb, uint32_t x) {
  if (cb == 2) {
    // v_sad_u8(x, 0, 0x6400) = 0x6400 + the sum of x's four bytes (each
    // |byte - 0|) in one instruction; 0x6400 + bsum is the fp16 encoding of
    // 1024 + bsum (bsum <= 1020). One fused fp16 FMA.
    const uint32_t h = __builtin_amdgcn_sad_u8(x, 0u, 0x6400u);
    return __builtin_fmaf16(f16_bits(h), f16_bits(0x1EEEu), f16_bits(0xC931u));
  }
  x = (x & 0x8FFF8FFFu) ^ 0x3B603B60u;
  return f16_bits(x & 0xFFFFu) + f16_bits(x >> 16);
}

// fp16 value of state s.
__device__ __forceinline__ f16 decode_state(int cb, uint32_t s) {
  return decode_hash(cb, hash_state(cb, s));
}
