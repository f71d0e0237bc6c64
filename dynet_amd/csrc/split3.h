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
// keep subnormal inputs and results.
//
// Infinities, NaNs, operands from 2^111 on and sums from 2^96 on come out as non-finite sums.  A wavefront that finds one
// among its sums of a 32 x 32 tile forms that tile again over its part of the depth with the fp32 instruction, from memory
// (add_products_fp32), so that infinities keep their sign and huge values their value.  A product full of NaNs takes two to
// seven times as long as one of numbers: 10 000 x 4480 x 1024 0.49 -> 3.2 ms, 2051 x 2050 x 650 0.07 -> 0.18 ms, 1024 x
// 512 x 784 16 -> 34 us (fp32 instruction alone: 0.71, 0.13 ms and 29 us; each output by itself, one multiply-add after
// another: 97, 3.6 and 0.34 ms); one NaN in the first 1.1 ms.
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

// The same parts, bit for bit, by shift, mask and subtraction: 13 instructions a pair.  The dot product instruction does
// not run beside matrix instructions (two wavefronts a SIMD, 16 of it and 4 products of 16 x 16 x 32: 214 cycles together,
// 96 and 81 apart; 16 multiplications and the same products 140), so where splits are dealt between products these are
// faster: 10 000 x 4480 x 1024 in 256 x 256 tiles 493 -> 483 us, 650 x 700 x 10 000 in 128 x 128 tiles 80.7 -> 78.7.
// Where a wavefront splits first and multiplies then they are not: 2048 x 2240 x 512 in gemm_direct.hip 48.7 -> 50.4.
__device__ __forceinline__ void split3_pair_beside_products(float a, float b, unsigned& h, unsigned& m, unsigned& l) {
  a *= kSplitIn;
  b *= kSplitIn;
  h = __builtin_bit_cast(unsigned, __builtin_convertvector(floatx2{a, b}, bf16x2));
  a -= __uint_as_float(h << 16);
  b -= __uint_as_float(h & 0xffff0000u);
  m = __builtin_bit_cast(unsigned, __builtin_convertvector(floatx2{a, b}, bf16x2));
  a -= __uint_as_float(m << 16);
  b -= __uint_as_float(m & 0xffff0000u);
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

typedef float sums16 __attribute__((ext_vector_type(16)));

// Whether any lane holds a sum that is infinite or NaN (0 times it is not 0).
template <typename T>
__device__ __forceinline__ bool any_not_finite(const T& x) {
  float z = 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r) z = fmaf(x[r], 0.f, z);
  return __any(!(z == 0.f));
}

// four values of a row, contiguous or ld apart
template <bool KMAJOR>
__device__ __forceinline__ float4 load4_fp32(const float* p, size_t ld) {
  typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));
  if (KMAJOR) {
    const float4u v = *reinterpret_cast<const float4u*>(p);
    return make_float4(v[0], v[1], v[2], v[3]);
  }
  const __attribute__((address_space(1))) float* q = (const __attribute__((address_space(1))) float*)p;
  float x[4];
#pragma unroll
  for (int c = 0; c < 4; ++c, q += ld) {
    asm volatile("" : "+v"(q));  // one address at a time: the registers are full of sums
    x[c] = *q;
  }
  return make_float4(x[0], x[1], x[2], x[3]);
}

// values `first` .. `first` + 3 of n, zeros from n on (read at the last one)
template <bool KMAJOR>
__device__ __forceinline__ float4 load4_fp32(const float* p, size_t ld, unsigned first, unsigned n) {
  float x[4];
#pragma unroll
  for (unsigned c = 0; c < 4; ++c) {
    const float v = p[min(first + c, n - 1) * (KMAJOR ? size_t(1) : ld)];
    x[c] = first + c < n ? v : 0.f;
  }
  return make_float4(x[0], x[1], x[2], x[3]);
}

__device__ __forceinline__ void mma8_fp32(sums16& sum, const float4& a, const float4& b) {
  sum = __builtin_amdgcn_mfma_f32_32x32x2f32(b.x, a.x, sum, 0, 0, 0);
  sum = __builtin_amdgcn_mfma_f32_32x32x2f32(b.y, a.y, sum, 0, 0, 0);
  sum = __builtin_amdgcn_mfma_f32_32x32x2f32(b.z, a.z, sum, 0, 0, 0);
  sum = __builtin_amdgcn_mfma_f32_32x32x2f32(b.w, a.w, sum, 0, 0, 0);
}

// sum += the products of depth k0 .. k1 - 1 of a 32 x 32 tile, where a and b are this lane's (l % 32) row of the left and
// column of the right operand; 32 k are fetched at a time.  mask: multiplies the row (stored along k, like it).
template <bool AK, bool BKM>
__device__ __forceinline__ void add_products_fp32(sums16& sum, const float* a, size_t lda, const float* b, size_t ldb,
                                                  unsigned k0, unsigned k1, const float* mask = nullptr) {
  const unsigned first = (threadIdx.x >> 3) & 4;  // lanes of the upper half take the second four of eight k
  const size_t sa = AK ? 1 : lda, sb = BKM ? 1 : ldb;
  a += size_t(k0) * sa;
  b += size_t(k0) * sb;
  if (mask != nullptr) mask += k0;
  unsigned left = k1 > k0 ? k1 - k0 : 0;
#pragma unroll 1
  for (; left >= 32; left -= 32) {
    float4 x[4], y[4];
#pragma unroll
    for (unsigned i = 0; i < 4; ++i, a += 8 * sa, b += 8 * sb) {
      x[i] = load4_fp32<AK>(a + first * sa, lda);
      y[i] = load4_fp32<BKM>(b + first * sb, ldb);
    }
    if (mask != nullptr) {
#pragma unroll
      for (unsigned i = 0; i < 4; ++i, mask += 8) {
        const float4 m = load4_fp32<true>(mask + first, 0);
        x[i] = make_float4(x[i].x * m.x, x[i].y * m.y, x[i].z * m.z, x[i].w * m.w);
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // every load under way before the first is waited for
#pragma unroll
    for (unsigned i = 0; i < 4; ++i) mma8_fp32(sum, x[i], y[i]);
  }
#pragma unroll 1
  for (; left > 0; left -= left < 8 ? left : 8, a += 8 * sa, b += 8 * sb) {
    float4 x = load4_fp32<AK>(a, lda, first, left);
    const float4 y = load4_fp32<BKM>(b, ldb, first, left);
    if (mask != nullptr) {
      const float4 m = load4_fp32<true>(mask, 0, first, left);
      mask += 8;
      x = make_float4(x.x * m.x, x.y * m.y, x.z * m.z, x.w * m.w);
    }
    mma8_fp32(sum, x, y);
  }
}

}  // namespace dyhip
