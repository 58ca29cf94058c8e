// Three bf16 terms of an f32 value and where they live in memory: shared by the kernels that write such planes.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace ughip {

// x = hi + mid + lo with every term a bf16 (round to nearest even of what the terms before left): 24 mantissa bits in
// three pieces, so |x - (hi + mid + lo)| <= 2^-25 |x|.  x3 row r holds, for every 64 columns c0 .. c0 + 63 of x, the
// three planes side by side: [hi(c0..) | mid(c0..) | lo(c0..)], i.e. K tile t of x3 is plane t % 3 of K tile t / 3 of x,
// and the three of them meet the same K tile of the matrix one after the other.
__device__ __forceinline__ uint16_t bf16_rne(float f) {
  const uint32_t x = __float_as_uint(f);
  if ((x & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((x >> 16) | 0x40u);  // NaN stays NaN
  return (uint16_t)((x + 0x7fffu + ((x >> 16) & 1u)) >> 16);
}
// Two values -> three words of two bf16 each (x0 in the low half); remainders are exact f32 subtractions.  An infinity (given, or
// reached when |x| rounds up past the largest bf16) or a NaN is all in the first term: the remainders would be inf - inf, and the
// product has to give what the f32 pipe gives for such an x (FINITE: the caller knows there is no infinity, e.g. among the
// exponentials of a softmax; a NaN then gives three NaNs).  The conversions round two values at once and branch nowhere: a norm
// of 1900 rows of 2048 to planes 9.7 -> 7.9 us, a gated fold of 1900 rows of 2 x 5632 36.2 -> 34.8 us against integer rounding with a branch
// for NaN.
typedef __bf16 split_bf16x2 __attribute__((ext_vector_type(2)));
typedef float split_f32x2 __attribute__((ext_vector_type(2)));
template <bool FINITE = false>
__device__ __forceinline__ void split3_pair(float x0, float x1, unsigned& hi, unsigned& mid, unsigned& lo) {
  const unsigned h = __builtin_bit_cast(unsigned, __builtin_convertvector(split_f32x2{x0, x1}, split_bf16x2));
  float r0 = x0 - __uint_as_float(h << 16), r1 = x1 - __uint_as_float(h & 0xffff0000u);
  if (!FINITE) {
    if ((h & 0x7f80u) == 0x7f80u) r0 = 0.f;
    if ((h & 0x7f800000u) == 0x7f800000u) r1 = 0.f;
  }
  const unsigned m = __builtin_bit_cast(unsigned, __builtin_convertvector(split_f32x2{r0, r1}, split_bf16x2));
  const float q0 = r0 - __uint_as_float(m << 16), q1 = r1 - __uint_as_float(m & 0xffff0000u);
  hi = h, mid = m, lo = __builtin_bit_cast(unsigned, __builtin_convertvector(split_f32x2{q0, q1}, split_bf16x2));
}

// Four consecutive elements of a row of k, split, to their places in the row's planes (x3_row: the row's first element).
__device__ __forceinline__ void split3_store4(const float in[4], uint16_t* __restrict__ x3_row, size_t col) {
  // the terms of the f32 value, as if it had been stored: a product in front of this must not be fused into the first remainder
  float x[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    x[i] = in[i];
    asm("" : "+v"(x[i]));
  }
  uint2 hi, mid, lo;
  split3_pair(x[0], x[1], hi.x, mid.x, lo.x);
  split3_pair(x[2], x[3], hi.y, mid.y, lo.y);
  uint16_t* o = x3_row + (col / 64) * 192 + col % 64;
  *reinterpret_cast<uint2*>(o) = hi;
  *reinterpret_cast<uint2*>(o + 64) = mid;
  *reinterpret_cast<uint2*>(o + 128) = lo;
}

}  // namespace ughip
