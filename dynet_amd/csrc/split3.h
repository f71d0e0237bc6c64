// fp32 products on the bf16 matrix cores.
//
// The fp32 matrix-core instructions run at 157 TFLOP/s on this part and the bf16 ones at 2.5 PFLOP/s.  An fp32 value is
// the sum of three bf16 values, x = h + m + l: h is x rounded to bf16, m the rest rounded to bf16, l what is left, and
// the three 8-bit significands hold all 24 bits of x.  A product x*y is then formed from six of the nine bf16 products,
//     l*h' + m*h' + m*m' + h*m' + h*l' + h*h',
// each exact in fp32, accumulated in fp32.  Rounding to nearest leaves |m| <= 2^-8 |x| and |l| <= 2^-17 |x|, so the
// three products left out (m*l', l*m', l*l') are at most (2^-25 + 2^-25 + 2^-34) |x y| together and typically a quarter
// of that: about the 2^-25 |x y| by which rounding an fp32 product is off at most.
//
// A matrix instruction rounds its accumulator once, however many of its 16 products are zero.  All six in one accumulator
// would round a long sum six times in 16 k, where fp32 arithmetic rounds once a product that is not zero: worse than fp32
// from half of the products zero on.  So the products h*h' have an accumulator of their own, and the five small ones,
// whose sums are 2^-8 of it, share another (gemm_wide.hip, which has no registers for that, forms each step's sum by
// itself).  Against fp64, K = 512, products that are not zero 100 / 25 / 10 / 1 %, in units of 1e-8:
//   one accumulator 17 / 15 / 12 / 6.5,  two 7.7 / 5.9 / 5.2 / 4.4,  the fp32 instruction 29 / 15 / 9.8 / 4.7.
//
// The smallest bf16 value is 2^-133, so the parts of x hold all of it only if its last bit is at least that: |x| >= 2^-110.
// fp32 values reach down to 2^-149 (probabilities of a confident softmax are that small), so every operand is multiplied
// by 2^16 on its way into the parts, exactly, and a sum by 2^-32 on its way out: all fp32 values are then split exactly,
// subnormals included (at 2^-120, unscaled, a product was off by 4e-5, below 2^-134 it was zero).  The bf16 instructions
// keep subnormal inputs and results.  Infinities, NaNs, operands from 2^111 on and sums from 2^96 on come out as
// non-finite sums; the kernels form such an output again with plain fp32 multiply-adds (dot_fp32), so that infinities
// keep their sign and huge values their value.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace dyhip {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx2 __attribute__((ext_vector_type(2)));

constexpr float kSplitIn = 65536.f;                // of an operand on its way into its parts
constexpr float kSplitOut = 1.f / (65536.f * 65536.f);  // of a sum of products of parts

// Two floats -> the bf16 parts of 2^16 times them, packed (first value in the low half): 9 instructions.  What is left of a value is the
// two-term dot product v + p.lo * s.lo + p.hi * s.hi with a selector s that takes one part of the pair away: one
// instruction where shift (or mask) and subtraction are two (11 instructions a pair; a loop of splits 1470 -> 1130 us).
// The difference is exact, subnormals included, so that the parts are the same bit for bit.  The other part is
// multiplied by -0: an infinity or NaN spreads to its neighbour, which feeds the same outputs.  (-0 and not 0: a
// selector that looks like the fp32 constant -1.0 would be encoded as one, whose low half is 0.)
__device__ __forceinline__ float take_away(unsigned parts, unsigned selector, float v) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, parts), __builtin_bit_cast(bf16x2, selector), v, false);
}

__device__ __forceinline__ void split3_pair(float a, float b, unsigned& h, unsigned& m, unsigned& l) {
  constexpr unsigned kLow = 0x8000BF80u, kHigh = 0xBF808000u;  // (-1, -0) and (-0, -1), low half first
  a *= kSplitIn;
  b *= kSplitIn;
  h = __builtin_bit_cast(unsigned, __builtin_convertvector(floatx2{a, b}, bf16x2));
  a = take_away(h, kLow, a);
  b = take_away(h, kHigh, b);
  m = __builtin_bit_cast(unsigned, __builtin_convertvector(floatx2{a, b}, bf16x2));
  a = take_away(m, kLow, a);
  b = take_away(m, kHigh, b);
  l = __builtin_bit_cast(unsigned, __builtin_convertvector(floatx2{a, b}, bf16x2));
}

// eight floats -> the fragments of the parts of 2^16 times them
struct Split3 {
  bf16x8 h, m, l;
  __device__ __forceinline__ void from(const float4& x, const float4& y) {
    uint4 ph, pm, pl;
    split3_pair(x.x, x.y, ph.x, pm.x, pl.x);
    split3_pair(x.z, x.w, ph.y, pm.y, pl.y);
    split3_pair(y.x, y.y, ph.z, pm.z, pl.z);
    split3_pair(y.z, y.w, ph.w, pm.w, pl.w);
    h = __builtin_bit_cast(bf16x8, ph);
    m = __builtin_bit_cast(bf16x8, pm);
    l = __builtin_bit_cast(bf16x8, pl);
  }
};

__device__ __forceinline__ bool not_finite(float x) { return !(x - x == 0.f); }
__device__ __forceinline__ bool not_finite(const float4& v) {
  return !((v.x - v.x) + (v.y - v.y) + (v.z - v.z) + (v.w - v.w) == 0.f);
}

// sum over k of a[k * step_a] * b[k * step_b], one multiply-add after another
__device__ __forceinline__ float dot_fp32(const float* a, size_t step_a, const float* b, size_t step_b, unsigned K) {
  float s = 0.f;
#pragma unroll 1
  for (unsigned k = 0; k < K; ++k) s = fmaf(a[size_t(k) * step_a], b[size_t(k) * step_b], s);
  return s;
}

}  // namespace dyhip
