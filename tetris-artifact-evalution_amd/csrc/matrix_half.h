// What the kernels that multiply fp16 parts (matrix_half.hip, matrix_relay.hip) share: how numbers are cut, the products, what a
// step's weights look like.
#pragma once
#include "matrix.h"

namespace tetris {
namespace {

typedef __bf16 bf16x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x8 __attribute__((ext_vector_type(8)));

// fp16 parts: an input times a power of two of the workgroup's is h + 2^-8 m + 2^-15 l, a weight times the power of two that
// brings the largest of its row to [2^14, 2^15) likewise.  h has eight bits, m eleven, l the rest.  (With 2^-19 l inputs of 2^-32
// of the largest would still be the sum of their parts, but of subnormal ones, whose left-out products are not small any more.)
constexpr float kMid = 256.f, kLow = 128.f;  // from h to m, from m to l
// Exponents of scaled inputs: the smallest that is multiplied in parts, from which on all 24 bits are in them; below the largest that
// h holds; the smallest that is listed where it is not, and above the largest.
constexpr float kRest = 2048.f;  // of a number in two parts: from the first to the second
constexpr int kSmall = -16, kSmall2 = -13, kLarge = 15, kLeastListed = -60, kMostListed = 40;

// (A bit cast of a vector's element itself, instead of its value, is compiled to one of the vector's first element.)
__device__ __forceinline__ float float_of(unsigned x) { return __builtin_bit_cast(float, x); }

// Three fp16 parts of eight floats, scaled; `zeros` becomes NaN where an h is infinite or NaN, `rest` (if any) gets a bit that is not
// zero where the parts do not add up to the floats.  (h is the bf16 number itself from 2^-16 of its scale on, so what is left of x
// takes full-rate FMAs; with inputs tested by `rest` and taken off h in fp16 workgroups were 1 % slower.)
__device__ __forceinline__ void cut16(const float (&x)[8], float scale, u32x4& hi, u32x4& mid, u32x4& lo, f16x2& zeros, unsigned* rest) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = x[2 * i], b = x[2 * i + 1];
    const unsigned t = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{a * scale, b * scale}), bf16x2));
    const float h0 = __builtin_bit_cast(float, t << 16), h1 = __builtin_bit_cast(float, t & 0xffff0000u);
    const f16x2 h = __builtin_convertvector((f32x2{h0, h1}), f16x2);
    const float r0 = fmaf(h0, -kMid, a * (scale * kMid)), r1 = fmaf(h1, -kMid, b * (scale * kMid));
    const f16x2 m = __builtin_convertvector((f32x2{r0, r1}), f16x2);
    const float s0 = fmaf((float)m.x, -kLow, r0 * kLow), s1 = fmaf((float)m.y, -kLow, r1 * kLow);
    const f16x2 l = __builtin_convertvector((f32x2{s0, s1}), f16x2);
    zeros = __builtin_elementwise_fma(h, f16x2{0, 0}, zeros);
    if (rest) *rest |= bits_of(fmaf((float)l.x, -1.f, s0)) | bits_of(fmaf((float)l.y, -1.f, s1));
    hi[i] = __builtin_bit_cast(unsigned, h);
    mid[i] = __builtin_bit_cast(unsigned, m);
    lo[i] = __builtin_bit_cast(unsigned, l);
  }
}

// From the parts of eight weights (the last one as it is kept, 2^-7 of it): `near`, the weights to eleven bits, `far`, 2^-7 of
// those, and `off`, what `near` is off by.  Subnormal roundings of fp16 cost a weight of 2^-3 or more (in its scale, where its
// row's largest is 2^14 or more) less than 2^-30 of it.
__device__ __forceinline__ void near_and_off(u32x4 hi, u32x4 mid, u32x4 lo, u32x4& near, u32x4& far, u32x4& off) {
  const f16x8 h = __builtin_bit_cast(f16x8, hi), m = __builtin_bit_cast(f16x8, mid);
  const f16x8 n = __builtin_elementwise_fma(m, (f16x8)(_Float16)(1 / kMid), h);
  near = __builtin_bit_cast(u32x4, n);
  far = __builtin_bit_cast(u32x4, n * (f16x8)(_Float16)(1 / kLow));
  u32x4 rest;  // h - near, which the compiler would take apart
#pragma unroll
  for (int i = 0; i < 4; ++i) asm("v_pk_add_f16 %0, %1, %2 neg_lo:[0,1] neg_hi:[0,1]" : "=v"(rest[i]) : "v"(hi[i]), "v"(near[i]));
  const f16x8 o = __builtin_elementwise_fma(__builtin_bit_cast(f16x8, rest), (f16x8)(_Float16)kMid, m);  // times 2^8, exactly
  const u32x4 o4 = __builtin_bit_cast(u32x4, o);
  u32x4 both;
#pragma unroll
  for (int i = 0; i < 4; ++i) asm("v_pk_add_f16 %0, %1, %2" : "=v"(both[i]) : "v"(o4[i]), "v"(lo[i]));
  off = __builtin_bit_cast(u32x4, __builtin_bit_cast(f16x8, both) * (f16x8)(_Float16)(1 / kMid));
}

// c + a * b: a 32 x 32, of which four consecutive values of a row hold two (`index` says which), b 32 x 32
template <bool F16>
__device__ __forceinline__ f32x16 product(u32x4 a, u32x4 b0, u32x4 b1, int index, f32x16 c) {
  const u32x8 b = __builtin_shufflevector(b0, b1, 0, 1, 2, 3, 4, 5, 6, 7);
  if constexpr (F16)
    return __builtin_amdgcn_smfmac_f32_32x32x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x16, b), c, index, 0, 0);
  else
    return __builtin_amdgcn_smfmac_f32_32x32x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x16, b), c, index, 0, 0);
}

// maximum over the wave
__device__ __forceinline__ unsigned wave_max(unsigned v) {
  auto step = [&](auto lanes) { v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, decltype(lanes)::value, 0xf, 0xf, true)); };
  step(std::integral_constant<int, 0x111>{});  // one, two, four and eight lanes down in a row of 16, then the rows
  step(std::integral_constant<int, 0x112>{});
  step(std::integral_constant<int, 0x114>{});
  step(std::integral_constant<int, 0x118>{});
  step(std::integral_constant<int, 0x142>{});
  step(std::integral_constant<int, 0x143>{});
  return __builtin_amdgcn_readlane(v, 63);
}

// x / d through magic_reciprocal(d), which is 0 for d = 1
__device__ __forceinline__ unsigned over(unsigned x, unsigned m) {
  const unsigned q = __umulhi(x, m);
  return m ? q : x;
}

// x / d for x below 2^30
__device__ __forceinline__ int quotient(int x, const MatDiv __attribute__((address_space(4)))& d) { return (int)((unsigned long long)(unsigned)x * d.m >> d.shift); }

// The weights of a step: three parts of eight slots per lane, then a word per lane (the slots' places in their groups of four,
// two bits each; above them the two blocks that the lane reads the input of).
static_assert(kStepBytes == 3 * 1024 + 256);

// Smallest weight, in its row's scale, that is kept in parts.  Smaller ones -- one in 10^5 of normally distributed weights -- are
// `loose`: multiplied one by one.  Where a block of 32 rows has more than kMostLoose, or one below kLeastLoose, whose
// products could underflow in the scale of the sums, the layer runs with bf16 parts.
constexpr float kLeast = 0x1p-3f, kLeastLoose = 0x1p-60f;
constexpr int kMostLoose = 64;

// Inputs that fp16 parts do not hold, or not well enough, are multiplied one by one as well: a wave stages zeros in their place and
// lists them, if they are 2^-60 to 2^40 in the tile's scale.  Where a workgroup has more than kMostAside, or others, it makes the second
// pass, and at once where a wave's first chunk already shows that.
constexpr unsigned kMostAside = 8, kNotListed = 1u << 24;
static_assert(kAsideBytes == 2 * 8 * 4 + 8 * 8 * kMostAside);  // of eight waves: counts after the first chunk and in the end, lists

struct MatArguments { const float* in; float* out; MatWeights w; MatGeom g; };
typedef const MatArguments __attribute__((address_space(4))) * Arguments;  // the kernel's, read through the scalar cache

}  // namespace
}  // namespace tetris
