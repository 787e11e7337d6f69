// fp32 products on the bf16 matrix cores: a float is split into three bf16 terms
// x = x0 + x1 + x2 (each the nearest bf16 of what the terms before it leave), and
// a b is the six products whose terms' orders add up to at most two,
//   a0 b0 + a0 b1 + a1 b0 + a0 b2 + a1 b1 + a2 b0,
// summed in the matrix cores' fp32 accumulators.  Three terms hold all 24
// significand bits; the dropped products are at most 2^-25 of |a b|, below
// the 2^-24 of the product's own fp32 rounding.  v_mfma_f32_32x32x16_bf16 has 16 times the
// fp32 MFMA's rate (32 cycles for 16 k against 64 for 2), so six of them are 2.7x
// as fast as the fp32 instruction, and one accumulator rounding covers 16
// products instead of 2.
//
// Range: the 24 bits hold for |x| from about 2^-109 (1.5e-33) on; below it the lower
// terms run into bf16's smallest values, 2^-133, whose halves are x's error.  An
// infinite operand, or one past bf16's largest value (3.39e38), which rounds to
// infinity, makes every sum it enters NaN (inf - inf in the split): a wave whose
// sums are not all finite (any_nonfinite) forms them again in fp32.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace ossm {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

// Eight k-consecutive values of one row (or column) as the three bf16 fragments
// of a 32x32x16 operand.
struct SplitFrag {
  bf16x8 t0, t1, t2;
};

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  const f32x2_t v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}
__device__ __forceinline__ float bf16_lo(uint32_t p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t p) { return __uint_as_float(p & 0xffff0000u); }

__device__ __forceinline__ SplitFrag split8(const float (&x)[8]) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  u32x4 p0, p1, p2;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = x[2 * i], b = x[2 * i + 1];
    p0[i] = pack_bf16(a, b);
    const float ra = a - bf16_lo(p0[i]), rb = b - bf16_hi(p0[i]);
    p1[i] = pack_bf16(ra, rb);
    p2[i] = pack_bf16(ra - bf16_lo(p1[i]), rb - bf16_hi(p1[i]));
  }
  return {__builtin_bit_cast(bf16x8, p0), __builtin_bit_cast(bf16x8, p1), __builtin_bit_cast(bf16x8, p2)};
}

__device__ __forceinline__ floatx16 mfma_bf16(bf16x8 a, bf16x8 b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Whether any sum that the wave holds is infinite or NaN (wave-uniform): their sum
// then is too (as where it overflows).
template <int N>
__device__ __forceinline__ bool any_nonfinite(const floatx16 (&c)[N]) {
  float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r & 3] += c[i][r];
  s[0] = (s[0] + s[1]) + (s[2] + s[3]);
  return __any(s[0] - s[0] != 0.f);
}

// c += a b over 2 k in fp32: lane l gives row (column) l % 32 at k = l / 32; the sums
// lie as the bf16 instruction's do.
__device__ __forceinline__ floatx16 mfma32(float a, float b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// c += a b over 16 k, smallest terms first
__device__ __forceinline__ floatx16 mfma_split(const SplitFrag& a, const SplitFrag& b, floatx16 c) {
  c = mfma_bf16(a.t2, b.t0, c);
  c = mfma_bf16(a.t1, b.t1, c);
  c = mfma_bf16(a.t0, b.t2, c);
  c = mfma_bf16(a.t1, b.t0, c);
  c = mfma_bf16(a.t0, b.t1, c);
  return mfma_bf16(a.t0, b.t0, c);
}

}  // namespace ossm
