// fp32 products on the bf16 matrix cores: x = hi + mid + lo with three bf16 parts (gfx950).
//
// Rounding to nearest even leaves |x - hi| <= 2^-9 |x| and |x - hi - mid| <= 2^-17 |x|, both
// differences exact in fp32 and the last one exact in bf16, so the three parts hold all 24
// significand bits of a number of at least 2^-110 (bf16 ends at 2^-133).  Of the nine products of
// two such numbers the six of at least 2^-18 are kept; the dropped ones are below 2^-25 of the
// product, unsigned bias included, against the 2^-24 of one fp32 rounding.  hi hi goes to one accumulator and the five corrections to
// another, so the small terms are not rounded away against a large sum.  Six
// v_mfma_f32_16x16x32_bf16 take 96 cycles where the eight v_mfma_f32_16x16x4_f32 they replace
// take 256.
//
// Infinities, NaN and magnitudes that round past bf16's largest number give a non-finite part
// and so a non-finite sum, also where the fp32 product is finite (inf * 0 of a zero part).
// Callers form every non-finite result again in plain fp32; products also those so small that
// numbers below 2^-110 may have made them (split_holds).  Attention does not: its weights are at
// most 1, and one below 2^-110 is uncertain by 76 x 2^-24 already through the score in its exponent.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cg {

typedef __attribute__((ext_vector_type(8))) __bf16 split_bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 split_bf16x2;
typedef __attribute__((ext_vector_type(4))) unsigned int split_u32x4;
typedef __attribute__((ext_vector_type(2))) float split_f32x2;
typedef __attribute__((ext_vector_type(4))) float split_f32x4;

// The parts of eight consecutive values (one lane's MFMA operand of 32 k).
struct Split8 {
  split_u32x4 hi, mid, lo;
};

__device__ __forceinline__ unsigned split_pack(float a, float b) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector(split_f32x2{a, b}, split_bf16x2));
}

// Two values: their packed parts (a in the low half).
__device__ __forceinline__ void split_pair(float a, float b, unsigned &hi, unsigned &mid, unsigned &lo) {
  hi = split_pack(a, b);
  a -= __uint_as_float(hi << 16);
  b -= __uint_as_float(hi & 0xffff0000u);
  mid = split_pack(a, b);
  a -= __uint_as_float(mid << 16);
  b -= __uint_as_float(mid & 0xffff0000u);
  lo = split_pack(a, b);
}

__device__ __forceinline__ Split8 split8(const split_f32x4 &x, const split_f32x4 &y) {
  Split8 s;
  unsigned h, m, l;
  split_pair(x[0], x[1], h, m, l);
  s.hi[0] = h, s.mid[0] = m, s.lo[0] = l;
  split_pair(x[2], x[3], h, m, l);
  s.hi[1] = h, s.mid[1] = m, s.lo[1] = l;
  split_pair(y[0], y[1], h, m, l);
  s.hi[2] = h, s.mid[2] = m, s.lo[2] = l;
  split_pair(y[2], y[3], h, m, l);
  s.hi[3] = h, s.mid[3] = m, s.lo[3] = l;
  return s;
}

__device__ __forceinline__ split_f32x4 split_mma1(const split_u32x4 &a, const split_u32x4 &b, const split_f32x4 &c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(split_bf16x8, a),
                                                 __builtin_bit_cast(split_bf16x8, b), c, 0, 0, 0);
}

// sum += a b over 32 k: the leading product into `acc`, the corrections into `cor`.
__device__ __forceinline__ void split_mma(const Split8 &a, const Split8 &b, split_f32x4 &acc, split_f32x4 &cor) {
  acc = split_mma1(a.hi, b.hi, acc);
  cor = split_mma1(a.lo, b.hi, cor);
  cor = split_mma1(a.hi, b.lo, cor);
  cor = split_mma1(a.mid, b.mid, cor);
  cor = split_mma1(a.mid, b.hi, cor);
  cor = split_mma1(a.hi, b.mid, cor);
}

__device__ __forceinline__ bool split_finite(float v) { return fabsf(v) <= 3.402823466e38f; }

// Whether a product's result stands: zero, or finite and at least 2^-80 (numbers below 2^-110 take a
// factor of 2^30 to reach that, and then an error of at most 2^-104).
constexpr unsigned SPLIT_LEAST = 0x17800000u, SPLIT_INF = 0x7f800000u;  // 2^-80, infinity
__device__ __forceinline__ bool split_holds(float v) {
  const unsigned u = __float_as_uint(v) & 0x7fffffffu;
  return (u - SPLIT_LEAST < SPLIT_INF - SPLIT_LEAST) | (u == 0);  // (no branch)
}

// A long sum with the rounding errors of its additions carried beside it (Knuth's two-sum): a bias
// gradient adds tens of thousands of rows, hundreds of them in one thread, and a result that is formed
// again (below) has one thread add all of k.
struct CarriedSum {
  float sum = 0.f, lost = 0.f;
  __device__ __forceinline__ void add(float x) {
#pragma clang fp contract(off) reassociate(off)
    const float s = sum + x, b = s - sum;
    lost += (sum - (s - b)) + (x - b);
    sum = s;
  }
  __device__ __forceinline__ float value() const { return split_finite(lost) ? sum + lost : sum; }  // (infinities)
};

}  // namespace cg
