// Floats as sums of bf16 parts for the bf16 matrix pipe, and the layout of staged rows of such parts.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace rpu_amd {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4_unaligned __attribute__((ext_vector_type(4), aligned(4))); // a 16-byte load from any float address

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Offset (in bf16) of 16-byte chunk `chunk` (8 values, 0 .. 3) of staged input row `row`: four rows of 64 bytes fill a
// 256-byte line, and the rotation by row / 4 lets 16 rows that read the same chunk touch all 64 banks once.
__device__ __forceinline__ int big_x_offset(int row, int chunk) {
  return (row >> 2) * 128 + (((row & 3) << 2) + ((chunk + (row >> 2)) & 3)) * 8;
}

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// Both rounded to nearest even.  For an MFMA by an instruction that the compiler chooses: an MFMA must not read a register
// sooner than two wait states after a vector instruction wrote it, and the compiler does not see that in assembly text (the
// second register of an operand that was converted one instruction before came out stale).  The empty text keeps it from
// rounding the value a second time where the halves are widened again.  STAGED: for LDS, where the hardware waits; as
// assembly text, which the compiler leaves closer to the store (three parts, 64 x 64 tiles, 1024 x 1024 backward: batch 1024
// 47.0 -> 39.6 us, batch 2048 56.1 -> 53.9).
template <bool STAGED> __device__ __forceinline__ uint32_t pack_bf16(float lower, float upper) {
  if (STAGED) {
    uint32_t p;
    asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(p) : "v"(lower), "v"(upper));
    return p;
  }
  uint32_t p = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lower, upper}, bf16x2));
  asm("" : "+v"(p));
  return p;
}
// v = hi + mid + lo with every part rounded to bf16: 3 x 8 bits hold the 24 of a float, so the sum is exact where the last
// bit of v is one that a bf16 can have, 2^-133.  The last bit of a float may be 2^-149: the kernel splits 2^16 times the
// value.
template <bool STAGED> __device__ __forceinline__ void split_bf16(const f32x4 v, u32x2 &hi, u32x2 &mid, u32x2 &lo) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float a = v[2 * i], b = v[2 * i + 1];
    hi[i] = pack_bf16<STAGED>(a, b);
    const float a1 = a - __uint_as_float(hi[i] << 16), b1 = b - __uint_as_float(hi[i] & 0xffff0000u);
    mid[i] = pack_bf16<STAGED>(a1, b1);
    lo[i] = pack_bf16<STAGED>(a1 - __uint_as_float(mid[i] << 16), b1 - __uint_as_float(mid[i] & 0xffff0000u));
  }
}
// Values of two operands, both split as 2^16 times themselves, below which the sum of `terms` of their products is finite before the
// 2^32 is taken out of it: terms * safe^2 * 2^32 <= 2^127.  The largest power of two that is.
__host__ __device__ inline float parts_safe(int terms) {
  const int bits = terms > 1 ? 32 - __builtin_clz((unsigned)terms - 1u) : 0;
  return __builtin_bit_cast(float, (uint32_t)(127 + (95 - bits) / 2) << 23);
}
__device__ __forceinline__ float max_abs4(float m, const f32x4 v) { // NaN do not count
  // two instructions; the compiler quiets every operand of fmaxf first, eight more
  asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(m) : "v"(v.x), "v"(v.y));
  asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(m) : "v"(v.z), "v"(v.w));
  return m;
}

} // namespace rpu_amd
