// Convolution of a sparse filter on the matrix cores with their 2:4 sparse instructions, for layers where that is faster than the
// dense products of matrix_conv.hip.
//
// matrix_conv.hip multiplies zeros and all, eight bf16 products to an fp32 one.  Two things make that less here.
//   * Products: six.  An fp32 number is the sum of three fp16 ones, h + 2^-8 m + 2^-15 l, with 8, 11 and 11 bits.  h has only 8
//     so that h times h has 16: sums of such products are rounded hardly ever, which is what keeps the whole as exact as bf16
//     parts do.  With eleven bits in h an output was off twice as far (1.9e-7 of the largest against 1.0e-7, 16 x 128 channels
//     3x3).  To need six products nevertheless, a weight is also written as near + off, eleven bits and the rest, made in
//     registers from its parts: h xh + 2^-8 (m xh + l xh + off xm + near xm + near xl).  What that leaves out, off xl, is less than
//     2^-29.5 of the product, of the smallest inputs that are multiplied so (below) 2^-28.
//   * k-values: v_smfmac takes a left operand of which two in four consecutive k-values are kept, at the rate of a dense
//     product of half as many (32 cycles for 32 x 32 x 32, measured: 3.3 PFLOP/s of what it stands for, 1.7 dense).  Blocks --
//     one tap of 8 channels for 32 output channels -- with three or four weights in a group of four come twice, blocks of
//     zeros not at all; four blocks are a step.  A list made with the plan says which.
// One step of 32 k-values and 32 x 32 outputs so costs 192 cycles of a matrix core, where dense bf16 products cost 512.  Of layers
// whose filters are 80 to 95 % zeros it takes 1.1 to 2 blocks per block.
//
// Workgroup: KW teams of WM x WN waves on one tile of 32*WM output channels x 32*NB*WN output pixels.  Input is staged as in
// matrix_conv.hip, the three parts of a pixel side by side: which 8 channels of which tap a lane reads, the step's word says.
// Weights go from L2 to registers, three steps ahead (two where registers do not hold more): the waits are counted, and a
// barrier comes once per chunk of up to 64 channels only.
//
// What bounds it: issue and latency of a wave's own steps, 1.5 to 2 times what the matrix cores need (they are busy 0.43 to 0.46
// of the time); for small layers the start, 5400 cycles, in which arguments, lists and input arrive one after the other.
// Microseconds, matrix_conv.hip's best against this, the walk in brackets: 16 x 128 -> 128 28x28 3x3 of 85 % zeros 30.3, 23.8
// (31.3); 16 x 256 -> 256 28x28 to 14x14 of 85 % 44.9, 33.9 (45.0); 4 x 256 -> 256 28x28 of 90 % 35.3, 25.9 (33.3); 16 x 256 ->
// 512 26x26 of 85 % 148, 103 (125) -- of 226 tiles of 96 pixels; 170 of 128 pixels leave a third of the CUs idle: 125.
//
// Range: inputs are scaled by what a few of them, the same for all waves, show.  Inputs 2^6 times as large as those, or smaller than
// 2^-25 of the largest of them and not zero, are staged as zeros and multiplied one by one with FMAs in the end, up to eight of a workgroup.
// Where they are more, or infinite, it makes a second pass with bf16 parts, which hold every number (see matrix_conv.hip for those,
// and for what is out of their range: the third pass).  An input's size decides, and not whether its parts add up to it:
// with few significant bits they do so far below, where m has lost bits to fp16's smallest exponent, l carries the number, and off xl
// is 2^-17 of the product and more.  Weights that fp16 parts do not hold are few: FMAs add them at the end as well.
// Single inputs out of range are ordinary: one in 10^7 of normally distributed ones is below 2^-25 of the largest, which is one
// workgroup or two of 226 on 256 channels, and a launch ends with its slowest.  Microseconds with a second pass for each such workgroup
// and now, in brackets the walk: 16 x 256 -> 512 26x26 of 85 % zeros, channels that differ in scale by e^(normal) 198, 106 (124); SiLU of
// normal inputs 123, 112; softmax over the channels, where the first chunk shows that they are many, 246, 147; exp(3 normal) 245, 229.
// Testing and listing costs 0 to 0.35 us a launch.
#include <algorithm>
#include <cmath>
#include <numeric>

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
constexpr int kSmall = -16, kLarge = 15, kLeastListed = -60, kMostListed = 40;

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

// One pass over a tile of outputs.  0: with fp16 parts; false: some input (or the weights) cannot be written so, and nothing was
// stored.  1: with bf16 parts; false: some sum of the wave's is not finite.  2: the wave's outputs with FMAs.
template <int PASS, int WM, int WN, int NB, int KW, int TM>
__device__ __forceinline__ bool matrix_pass(Arguments arguments, int thread) {
  constexpr bool F16 = PASS == 0;
  constexpr int TW = WM * WN, P = 32 * NB * WN;
  const auto& g = arguments->g;
  // What the places of the pixels are worked out with, read at once: each first touch of a line is a trip to L2.
  const struct { unsigned m_uw, m_uh, m_wp, m_ihs, m_strips; int upq, uw, uh, wp, ihs, strips, ws, stride, sub, pad, pool, npix, H, W, C, N, ks, kgs, lpad; } at = {
      g.m_uw, g.m_uh, g.m_wp, g.m_ihs, g.m_strips, g.upq, g.uw, g.uh, g.wp, g.ihs, g.strips, g.ws, g.stride, g.sub, g.pad, g.pool, g.npix, g.H, g.W, g.C, g.N, g.ks, g.kgs, g.lpad};
  const auto& w = arguments->w;
  const float* const in = arguments->in;
  extern __shared__ u32x4 all_lds[];  // [KW][2][kgs][lpad][3], then the exponents of the tile's rows
  const int lane = thread & 63, wave_id = __builtin_amdgcn_readfirstlane(thread >> 6);
  const int team = wave_id / TW, wave = wave_id % TW;
  u32x4* const lds = all_lds + team * 6 * g.kgs * g.lpad;
  int* const row_exp = reinterpret_cast<int*>(reinterpret_cast<char*>(all_lds) + g.lds_rows);
  unsigned* const asides = reinterpret_cast<unsigned*>(row_exp + 32 * WM);  // per wave: how many inputs are set aside
  int2* const aside = reinterpret_cast<int2*>(asides + 16);                 // ... which: channel and staged pixel; the input
  // workgroup ids go round-robin to the XCDs: each XCD gets a contiguous range of logical ids.  Channel blocks of one pixel
  // tile are neighbours (they read the same input), slices outermost (they share nothing).
  const int per = gridDim.x >> 3;
  const int id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  const int tiles = g.ptiles * g.mtiles;
  const int slice = quotient(id, g.d_tiles), tile = id - slice * tiles;
  const int pt = quotient(tile, g.d_mtiles), mt = tile - pt * g.mtiles;
  const int wm = wave % WM, wn = wave / WM;
  const int block = min(mt * WM + wm, g.mblocks - 1);

  // first pixel of the tile: strip image q0, row and column in it (in 2x2 blocks when pooling)
  const int psh = g.pool ? 2 : 0, dbl = g.pool ? 1 : 0;
  const int u0 = (pt * P) >> psh;
  const int q0 = quotient(u0, g.d_upq), r0 = u0 - q0 * g.upq;
  const int oy0 = quotient(r0, g.d_uw), ox0 = r0 - oy0 * g.uw;
  const int row0 = (oy0 << dbl) * g.stride, col0 = (ox0 << dbl) * g.stride;

  // the teams of a workgroup share the slice's chunks, at least one each
  const int s_beg = slice * g.chunks / g.csplit, s_len = (slice + 1) * g.chunks / g.csplit - s_beg;
  const int c_beg = s_beg + s_len * team / KW, mine = s_beg + s_len * (team + 1) / KW - c_beg, rounds = (s_len + KW - 1) / KW;

  // Weights: the steps of a wave follow one another; they are asked for three steps ahead of their products.
  struct Step { u32x4 p[F16 ? 3 : 2]; unsigned word; };
  int next_step = w.first[block * g.chunks + c_beg];
  const int loose = F16 ? w.loose_count[block] : 0, steps = w.first[block * g.chunks + c_beg + mine] - next_step;
  const __amdgpu_buffer_rsrc_t wrsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(w.steps), 0, w.step_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t srsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(w.slots), 0, w.step_bytes / kStepBytes * kSlotBytes, 0x00020000);
  auto fetch_weights = [&](Step& s) {
#pragma unroll
    for (int p = 0; p < (F16 ? 3 : 2); ++p)
      s.p[p] = __builtin_amdgcn_raw_buffer_load_b128(F16 ? wrsrc : srsrc, lane * 16 + p * 1024, next_step * (F16 ? kStepBytes : kSlotBytes), 0);
    s.word = __builtin_amdgcn_raw_buffer_load_b32(wrsrc, lane * 4 + 3072, next_step * kStepBytes, 0);
    ++next_step;
  };

  // what this wave stages: 64 staged pixels of one channel group per task
  const int blocks = g.lpad >> 6, tasks = g.kgs * blocks;
  int goff[TM], gkg[TM], gslot[TM];
#pragma unroll
  for (int k = 0; k < TM; ++k) {
    const int task = wave + TW * k;
    gkg[k] = quotient(task, g.d_blocks);
    const int blk = task - gkg[k] * blocks;
    gslot[k] = 3 * (gkg[k] * at.lpad + blk * 64 + lane);
    const unsigned x = col0 + blk * 64 + lane;
    const unsigned dr = over(x, at.m_wp), col = x - dr * at.wp;
    const unsigned row = row0 + dr;
    const unsigned dq = over(row, at.m_ihs), y = row - dq * at.ihs;
    const unsigned q = q0 + dq, n = over(q, at.m_strips), strip = q - n * at.strips;
    const int iy = (int)y * at.sub - at.pad, ix = (int)(strip * at.ws * at.stride + col) * at.sub - at.pad;
    goff[k] = task < tasks && n < (unsigned)at.N && iy >= 0 && iy < at.H && ix >= 0 && ix < at.W
                  ? 4 * (int)(n * (unsigned)(at.C * at.H * at.W) + (unsigned)(iy * at.W + ix)) : kOutside;
  }
  const int hw4 = 4 * g.H * g.W;
  const __amdgpu_buffer_rsrc_t irsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(in), 0, g.in_bytes, 0x00020000);
  float x[TM][8];
  auto fetch = [&](int chunk) {
#pragma unroll
    for (int k = 0; k < TM; ++k) {
      if (wave + TW * k >= tasks) break;
      const int c = (chunk * at.kgs + gkg[k]) * 8;
      if (c + 8 <= at.C) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
          x[k][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(irsrc, goff[k], (c + j) * hw4, 0));
      } else {  // channels that do not exist are zero
#pragma unroll
        for (int j = 0; j < 8; ++j)
          x[k][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                  irsrc, c + j < at.C ? goff[k] : kOutside, min(c + j, at.C - 1) * hw4, 0));
      }
    }
  };
  float scale = 1.f;
  // the exponent bits of 2^e in the tile's scale, of a number that is not scaled yet (where it may underflow)
  auto unscaled = [&](int e) { return (unsigned)min(max(2 * 127 + e - (int)(bits_of(scale) >> 23), 0), 255) << 23; };
  // inputs of a lane that six products cannot be formed of: listed, and zero in its parts
  unsigned own_asides = loose < 0 ? kNotListed : 0;
  auto set_aside = [&](const float (&x)[8], u32x4& h, u32x4& m, u32x4& l, int slot, int channel) {
    unsigned which = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const unsigned u = bits_of(x[j]) & 0x7fffffff;
      if (u - 1 < unscaled(kSmall) - 1 || u >= unscaled(kLarge)) which |= 1u << j;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned held = (which >> 2 * i & 1 ? 0 : 0xffffu) | (which >> 2 * i & 2 ? 0 : 0xffff0000u);
      h[i] &= held;
      m[i] &= held;
      l[i] &= held;
    }
    while (const unsigned long long lanes = __builtin_amdgcn_ballot_w64(which != 0)) {
      const int j = __builtin_ctz(which | 256);
      float v = x[0];
#pragma unroll
      for (int q = 1; q < 8; ++q) v = j == q ? x[q] : v;
      const unsigned u = bits_of(v) & 0x7fffffff, n = own_asides + __builtin_amdgcn_mbcnt_hi(lanes >> 32, __builtin_amdgcn_mbcnt_lo(lanes, 0));
      const bool listed = u >= unscaled(kLeastListed) && u < unscaled(kMostListed);
      if (which && n < kMostAside) aside[wave_id * kMostAside + n] = make_int2((channel + j) << 10 | slot, (int)bits_of(v));
      own_asides = min(own_asides + (__builtin_amdgcn_ballot_w64(which && !listed) ? kNotListed : __builtin_popcountll(lanes)), kNotListed);
      which &= which - 1;
    }
  };
  auto keep = [&](int buf, int chunk) {
#pragma unroll
    for (int k = 0; k < TM; ++k) {
      if (wave + TW * k >= tasks) break;
      u32x4 h, m, l;
      if constexpr (F16) {
        f16x2 zeros = {0, 0};
        cut16(x[k], scale, h, m, l, zeros, nullptr);
        unsigned least = ~0u;  // of the inputs' bits without the sign, doubled, less one: zeros come out on top
#pragma unroll
        for (int j = 0; j < 8; ++j) least = min(least, (bits_of(x[k][j]) << 1) - 1);
        const bool infinite = __builtin_bit_cast(unsigned, zeros) & 0x7fff7fff;
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(infinite || least < 2 * unscaled(kSmall) - 1) != 0, 0))
          set_aside(x[k], h, m, l, gslot[k] / 3 - gkg[k] * at.lpad, (chunk * at.kgs + gkg[k]) * 8);
      } else {
        cut(x[k], h, m, l);
      }
      u32x4* d = lds + buf * 3 * at.kgs * at.lpad + gslot[k];
      d[0] = h;
      d[1] = m;
      d[2] = l;
    }
  };

  // The first input and the first weights are asked for before anything that they do not depend on is computed; before them
  // a few values from all over the tile's input, the same in all waves, which tell what it has to be scaled by.
  unsigned some[4];
  if constexpr (F16) {
    // (Sixteen neighbours of each of sixteen channels from all over the slice: a channel may be zero throughout, and their scales
    // differ.  With 64 of each of four, the last layer of a chain of VGG19's at batch 1 made both passes: 21.4 us, 11.9 so.)
    const int hw = at.H * at.W, from = max((int)(row0 - over(row0, at.m_ihs) * at.ihs) * at.sub - at.pad, 0) * at.W + (lane & 15);
    const int ch0 = s_beg * 8 * at.kgs, channels = min(s_len * 8 * at.kgs, at.C - ch0), image = 4 * (int)over(q0, at.m_strips) * at.C * hw;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      some[j] = __builtin_amdgcn_raw_buffer_load_b32(
          irsrc, image + 4 * min(from + (at.lpad * j >> 2), hw - 1) + (ch0 + (channels * (lane >> 4 << 2 | j) >> 4)) * hw4, 0, 0);
  }
  const int exponent = F16 ? w.row_exp[min(mt * WM * 32 + (thread & (32 * WM - 1)), 32 * g.mblocks - 1)] : 0;
  fetch(c_beg);

  // where this lane's pixels lie: in the output's images, in LDS and in the output
  struct Pixel { bool in_range; int t; unsigned n, dq, uy, oy, ox, w; };  // ox: in its strip, w: in its image
  auto pixel = [&](int b, int lane) {
    Pixel p;
    const int t = (wn * NB + b) * 32 + (lane & 31);
    p.in_range = pt * P + t < g.npix;
    p.t = p.in_range ? t : g.npix - 1 - pt * P;
    const unsigned x = ox0 + (p.t >> psh);
    const unsigned dy = over(x, at.m_uw), ux = x - dy * at.uw, y = oy0 + dy;
    p.dq = over(y, at.m_uh);
    p.uy = y - p.dq * at.uh;
    p.oy = (p.uy << dbl) + (at.pool ? (p.t >> 1) & 1 : 0);
    p.ox = (ux << dbl) + (at.pool ? p.t & 1 : 0);
    const unsigned q = q0 + p.dq;
    p.n = over(q, at.m_strips);
    p.w = (q - p.n * at.strips) * at.ws + p.ox;
    return p;
  };
  int bpos[NB], ooff[NB];
  const int ohw = g.pool ? (g.OH >> 1) * (g.OW >> 1) : g.OH * g.OW;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const Pixel p = pixel(b, lane);
    bpos[b] = 3 * (((int)(p.dq * g.ihs + p.oy * g.stride) - row0) * g.wp + (int)p.ox * g.stride - col0);
    if (g.pool)
      ooff[b] = p.in_range && (p.t & 3) == 0 && (p.w >> 1) < (unsigned)(g.OW >> 1)
                    ? 4 * (int)((p.n * g.K + 4 * (lane >> 5)) * ohw + p.uy * (g.OW >> 1) + (p.w >> 1)) : kOutside;
    else
      ooff[b] = p.in_range && p.w < (unsigned)g.OW ? 4 * (int)((p.n * g.K + 4 * (lane >> 5)) * ohw + p.oy * g.OW + p.w) : kOutside;
  }

  float* dst = arguments->out + (size_t)slice * g.out_floats;
  const __amdgpu_buffer_rsrc_t orsrc = __builtin_amdgcn_make_buffer_rsrc(dst, 0, 4 * g.out_floats, 0x00020000);
  const int oc0 = (mt * WM + wm) * 32;
  // sum i of a lane: channel 8*(i/4) + 4*(lane/32) + i%4 of its wave's 32, pixel lane%32
  auto store = [&](int i, int b, float v) {
    const int oc = oc0 + 8 * (i / 4) + i % 4;
    if (g.pool) v = quad_max(v);
    if (g.relu) v = fmaxf(v, 0.f);
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, v), orsrc, oc + 4 * (lane >> 5) < g.K ? ooff[b] : kOutside, oc * ohw * 4, 0);
  };
  if constexpr (PASS == 2) {
    // Latency of the loads bounds this, and it is here to be right.
    const int ch0 = slice * g.chunks / g.csplit * 8 * g.kgs, ch1 = min(g.C, (slice + 1) * g.chunks / g.csplit * 8 * g.kgs);
    const int cpad = 8 * g.kgs * g.chunks;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const Pixel p = pixel(b, lane);
      float sums[16 / KW];
#pragma unroll
      for (int j = 0; j < 16 / KW; ++j) sums[j] = 0;
#pragma nounroll
      for (int c = ch0; c < ch1; c += 8)
#pragma nounroll
        for (int r = 0; r < g.ks; ++r)
#pragma nounroll
          for (int s = 0; s < g.ks; ++s) {
            const int iy = (int)(p.oy * g.stride + r) * g.sub - g.pad, ix = (int)(p.w * g.stride + s) * g.sub - g.pad;
            const bool inside = iy >= 0 && iy < g.H && ix >= 0 && ix < g.W && p.n < (unsigned)g.N;
            const int at = 4 * (int)(((p.n * g.C + c) * g.H + iy) * g.W + ix);
            float v[8];
#pragma unroll
            for (int q = 0; q < 8; ++q)
              v[q] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                   irsrc, inside && c + q < g.C ? at + q * hw4 : kOutside, 0, 0));
#pragma unroll
            for (int j = 0; j < 16 / KW; ++j) {
              const int i = team * (16 / KW) + j, oc = oc0 + 8 * (i / 4) + 4 * (lane >> 5) + i % 4;
              const u32x4* d = reinterpret_cast<const u32x4*>(w.dense + (((size_t)min(oc, g.K - 1) * g.ks + r) * g.ks + s) * cpad + c);
              const u32x4 d0 = d[0], d1 = d[1];
#pragma unroll
              for (int q = 0; q < 8; ++q) {
                const float f = float_of(q < 4 ? d0[q % 4] : d1[q % 4]);
                if (f != 0.f) sums[j] = fmaf(v[q], f, sums[j]);
              }
            }
          }
#pragma unroll
      for (int j = 0; j < 16 / KW; ++j) store(team * (16 / KW) + j, b, sums[j]);
    }
    return true;
  }

  // The leading products and the others, 2^-8 of them, so that what is small is summed before it is rounded.
  f32x16 sum[2][NB];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int i = 0; i < 16; ++i) sum[0][b][i] = sum[1][b][i] = 0.f;
  constexpr int kSets = F16 ? NB > 2 ? 2 : 3 : 1;
  Step ahead[kSets];
#pragma unroll
  for (int i = 0; F16 && i < kSets; ++i) {
    fetch_weights(ahead[i]);
    __builtin_amdgcn_sched_barrier(0);  // in this order: the loop waits for the first set only
  }
  if constexpr (F16) {
    // Their largest is scaled to [2^9, 2^10).  (To [2^11, 2^12), with 4 bits to spare above, channels that differ in scale often had more
    // than a few inputs too large: 150 us for the 106 named above.)
    unsigned most = max(max(some[0] & 0x7fffffff, some[1] & 0x7fffffff), max(some[2] & 0x7fffffff, some[3] & 0x7fffffff));
    most = wave_max(most);
    const int shift = most ? min(max(136 - (int)(most >> 23), -100), 100) : 6;
    scale = __builtin_bit_cast(float, (127 + shift) << 23);
    if (thread < 32 * WM) row_exp[thread] = exponent - shift;
  }
  keep(0, c_beg);
  if (F16) asides[8 + wave_id] = own_asides > kMostAside || (own_asides > 2 && own_asides * (unsigned)rounds > kMostAside);
  __syncthreads();
  const int wp3 = 3 * at.wp, lpad3 = 3 * at.lpad;
  const bool large = at.ks > 4;
  int buf = 0, round = 0;
  bool fresh = true;  // the chunk's first step
  // A step reads the input of its two blocks of pixels one after the other, each while the products of the one before run: the
  // first block's while those of the step before do, unless a barrier lies between.
  int place[2];  // of the step's input: the blocks in the two halves of a lane's registers
  auto place_of = [&](unsigned word) {
    const int from = buf * 3 * at.kgs * at.lpad;
    if (!large) {
      place[0] = from + (int)(__umul24(word >> 16 & 3, 3) + __umul24(word >> 18 & 3, wp3) + __umul24(word >> 20 & 7, lpad3));
      place[1] = from + (int)(__umul24(word >> 24 & 3, 3) + __umul24(word >> 26 & 3, wp3) + __umul24(word >> 28 & 7, lpad3));
    } else {
      place[0] = from + (int)(__umul24(word >> 16 & 7, 3) + __umul24(word >> 19 & 7, wp3) + __umul24(word >> 22 & 1, lpad3));
      place[1] = from + (int)(__umul24(word >> 24 & 7, 3) + __umul24(word >> 27 & 7, wp3) + __umul24(word >> 30 & 1, lpad3));
    }
  };
  struct Input { u32x4 v[2][3]; };
  auto read = [&](Input& in, int b) {
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int p = 0; p < 3; ++p) in.v[r][p] = lds[place[r] + bpos[b] + p];
  };
  Input input[2];
  if constexpr (F16) {
    place_of(ahead[0].word);
    read(input[0], 0);
    if (__builtin_amdgcn_ballot_w64(asides[8 + (lane & (TW * KW - 1))] != 0)) return false;
  }
  // Where a wave has an odd number of blocks, more than one, two steps take turns with the two places for a block's input.
  auto step = [&](Step& now, Step& next, auto turn) {
    constexpr int kFirst = NB > 1 && NB % 2 ? decltype(turn)::value % 2 : 0, kNext = (kFirst + (NB > 1 ? NB : 0)) % 2;
    if constexpr (!F16) {
      fetch_weights(now);
      place_of(now.word);
      read(input[0], 0);
    }
    const unsigned word = now.word;
    const bool last = __builtin_amdgcn_readfirstlane(word) >> 31, more = round + 1 < mine;
    if constexpr (NB > 1) read(input[1 - kFirst], 1);
    if constexpr (F16) __builtin_amdgcn_sched_barrier(0);
    u32x4 a[F16 ? 6 : 3];
    if constexpr (F16) {
#pragma unroll
      for (int p = 0; p < 3; ++p) a[p] = now.p[p];
      near_and_off(a[0], a[1], a[2], a[3], a[4], a[5]);
    } else {
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = float_of(now.p[j / 4][j % 4]);
      cut(v, a[0], a[1], a[2]);
    }
    // The products, smallest first.  Of bf16 parts all but low times low.  Of fp16 parts, with a weight w = h + m + l =
    // near + off: h h + m h + near m + l h + off m + near l.  That leaves out off l.
    auto products = [&](const Input& in, int b) {
      if constexpr (F16) {
        constexpr int pa[6] = {2, 0, 1, 5, 3, 4}, pb[6] = {0, 0, 0, 1, 1, 2}, to[6] = {1, 0, 1, 1, 1, 1};
#pragma unroll
        for (int t = 0; t < 6; ++t) sum[to[t]][b] = product<true>(a[pa[t]], in.v[0][pb[t]], in.v[1][pb[t]], (int)word, sum[to[t]][b]);
      } else {
        constexpr int pa[8] = {2, 1, 2, 1, 0, 1, 0, 0}, pb[8] = {1, 2, 0, 1, 2, 0, 1, 0};
#pragma unroll
        for (int t = 0; t < 8; ++t) sum[t < 7][b] = product<false>(a[pa[t]], in.v[0][pb[t]], in.v[1][pb[t]], (int)word, sum[t < 7][b]);
      }
    };
#pragma unroll
    for (int b = 0; b < (NB > 1 ? NB - 1 : 1); ++b) {
      products(input[(kFirst + b) % 2], b);
      if (b > 0 || NB > 2) {
        if constexpr (F16) __builtin_amdgcn_sched_barrier(0);
        if (b + 2 < NB) read(input[(kFirst + b) % 2], b + 2);
        if constexpr (F16) __builtin_amdgcn_sched_barrier(0);
      }
    }
    auto refill = [&]() {
      if constexpr (F16) {
        __builtin_amdgcn_sched_barrier(0);
        if (fresh && more) fetch(c_beg + round + 1);
        fresh = false;
        __builtin_amdgcn_sched_barrier(0);
        fetch_weights(now);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    if (!last) {
      if constexpr (F16) {
        __builtin_amdgcn_sched_barrier(0);
        place_of(next.word);
        read(input[kNext], 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (NB > 1) products(input[(kFirst + NB - 1) % 2], NB - 1);
      refill();
      return;
    }
    // the chunk's last
    if constexpr (NB > 1) products(input[(kFirst + NB - 1) % 2], NB - 1);
    refill();
    if (!F16 && more) fetch(c_beg + round + 1);  // (the second pass is rare: fewer registers instead of less waiting)
    if (more) keep(buf ^ 1, c_beg + round + 1);
    if (F16 && round + 1 == rounds) asides[wave_id] = own_asides;
    buf ^= 1;
    fresh = true;
    ++round;
    __syncthreads();
    if constexpr (F16) {
      place_of(next.word);
      read(input[kNext], 0);
    }
  };
  for (int left = steps; left > 0; left -= kSets) {
    step(ahead[0], ahead[1 % kSets], std::integral_constant<int, 0>{});
    // (Waiting for all loads when the steps run out costs nothing that matters, and tells the compiler that at the head of the
    // loop the first set's loads are the oldest.)
    if constexpr (kSets > 1) {
      if (left > 1) step(ahead[1], ahead[2 % kSets], std::integral_constant<int, 1>{});
      else __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    }
    if constexpr (kSets > 2) {
      if (left > 2) step(ahead[2], ahead[0], std::integral_constant<int, 2>{});
      else __builtin_amdgcn_s_waitcnt(0x0f70);
    }
  }
  if (round < rounds) {  // a team with a chunk less
    if (F16) asides[wave_id] = own_asides;
    __syncthreads();
  }
  if constexpr (F16) {
    const unsigned listed = asides[lane / kMostAside & (TW * KW - 1)];  // by the wave whose list this lane may read
    const unsigned long long some_listed = __builtin_amdgcn_ballot_w64(lane < TW * KW * (int)kMostAside && lane % kMostAside < listed);
    if (__builtin_popcountll(some_listed) > (int)kMostAside || __builtin_amdgcn_ballot_w64(listed > kMostAside)) return false;
    // the weights that fp16 parts do not hold: few blocks have any
    int again = lane;  // (unknown to the compiler, which would else keep the pixels' places in registers all the while)
    asm("" : "+v"(again));
    for (int e = 0; e < loose; ++e) {
      const int where = w.loose[kMostLoose * block + e].x, row = where & 31, r = where >> 5 & 7, s = where >> 8 & 7, c = where >> 11;
      const float weight = __builtin_bit_cast(float, w.loose[kMostLoose * block + e].y);
      const int chunk = c / (8 * at.kgs);
      if (chunk < c_beg || chunk >= c_beg + mine) continue;
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const Pixel p = pixel(b, again);
        const int iy = (int)(p.oy * at.stride + r) * at.sub - at.pad, ix = (int)(p.w * at.stride + s) * at.sub - at.pad;
        const bool inside = iy >= 0 && iy < at.H && ix >= 0 && ix < at.W && p.n < (unsigned)at.N && (again >> 5) == (row >> 2 & 1);
        const float v = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                            irsrc, inside ? 4 * (int)(((p.n * at.C + c) * at.H + iy) * at.W + ix) : kOutside, 0, 0)) * scale;
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (i == (row >> 3) * 4 + (row & 3)) sum[0][b][i] = fmaf(v, weight, sum[0][b][i]);
      }
    }
    // The inputs that are set aside, with the weights that are not among those, in the order of their places: sums do not depend on
    // who came first.
    if (some_listed) {
      const int2 own = some_listed >> again & 1 ? aside[again] : make_int2(0x7fffffff, 0);
      const int all = __builtin_popcountll(some_listed);
      int before = 0;
      for (unsigned long long left = some_listed; left; left &= left - 1) before += __builtin_amdgcn_readlane(own.x, __builtin_ctzll(left)) < own.x;
      const int shift = (int)(bits_of(scale) >> 23) - 127, cpad = 8 * at.kgs * g.chunks;
      for (int e = 0; e < all; ++e) {
        const int from = __builtin_ctzll(__builtin_amdgcn_ballot_w64(before == e));
        const int where = __builtin_amdgcn_readlane(own.x, from), c = where >> 10, chunk = c / (8 * at.kgs);
        if (chunk < c_beg || chunk >= c_beg + mine) continue;
        const float v = float_of(__builtin_amdgcn_readlane(own.y, from)) * scale;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          int tap = -1;  // of the lane's pixel that reads it
          for (int r = 0; r < g.ks; ++r) {
            const int s = 3 * (where & 1023) - bpos[b] - 3 * r * at.wp;
            if (s >= 0 && s < 3 * g.ks) tap = r * g.ks + s / 3;
          }
          if (!__builtin_amdgcn_ballot_w64(tap >= 0)) continue;
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int row = 8 * (i / 4) + 4 * (again >> 5) + i % 4, oc = oc0 + row;
            const float weight = tap >= 0 && oc < g.K ? w.dense[((size_t)oc * g.ks * g.ks + tap) * cpad + c] : 0.f;
            const float scaled = ldexpf(weight, -(row_exp[wm * 32 + row] + shift));
            sum[0][b][i] = fmaf(v, fabsf(scaled) >= kLeast ? scaled : 0.f, sum[0][b][i]);
          }
        }
      }
    }
  }

  auto total = [&](int i, int b) {
    if constexpr (F16) return fmaf(sum[1][b][i], 1 / kMid, sum[0][b][i]);
    else return sum[0][b][i] + sum[1][b][i];
  };
  float odd = 0;  // NaN once a sum of bf16 parts is infinite or NaN
  auto scale_of = [&](int i) { return *reinterpret_cast<const int4*>(row_exp + wm * 32 + 2 * i + 4 * (lane >> 5)); };
  constexpr bool kScales = F16 && KW == 1 && NB < 4;  // registers for all of them
  int4 scales[4];
#pragma unroll
  for (int i = 0; kScales && i < 4; ++i) scales[i] = scale_of(4 * i);
  auto finish = [&](int i, int b, float (&v)[4]) {  // sums i to i + 3
    if constexpr (F16) {
      const int4 e = kScales ? scales[i / 4] : scale_of(i);
      v[0] = ldexpf(v[0], e.x); v[1] = ldexpf(v[1], e.y); v[2] = ldexpf(v[2], e.z); v[3] = ldexpf(v[3], e.w);
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        odd = fmaf(v[k], 0.f, odd);
        v[k] *= kUnscale;
      }
    }
    if (g.quads) {
      // four pixels of a channel to a lane instead of four channels of a pixel: a store of 16 bytes instead of four
      transpose_quad(v, lane);
      u32x4 d;
#pragma unroll
      for (int k = 0; k < 4; ++k) d[k] = bits_of(g.relu ? fmaxf(v[k], 0.f) : v[k]);
      __builtin_amdgcn_raw_buffer_store_b128(d, orsrc, oc0 + 2 * i + 4 * (lane >> 5) + (lane & 3) < g.K && ooff[b] != kOutside ? ooff[b] + 4 * (lane & 3) * (ohw - 1) : kOutside,
                                             (oc0 + 2 * i) * ohw * 4, 0);
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) store(i + k, b, v[k]);
    }
  };
  if constexpr (KW == 1) {
#pragma unroll
    for (int i = 0; i < 16; i += 4)
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        float v[4] = {total(i, b), total(i + 1, b), total(i + 2, b), total(i + 3, b)};
        finish(i, b, v);
      }
  } else {
    // every team leaves its sums in LDS and adds a share of all of them
    constexpr int kTeam = TW * 1024 * NB;
    float* sums = reinterpret_cast<float*>(all_lds) + wave * 1024 * NB + lane;
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
      for (int b = 0; b < NB; ++b) sums[team * kTeam + (i * NB + b) * 64] = total(i, b);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; i += 4) {
      if (i / (16 / KW) != team) continue;
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          v[j] = sums[((i + j) * NB + b) * 64];
#pragma unroll
          for (int k = 1; k < KW; ++k) v[j] += sums[k * kTeam + ((i + j) * NB + b) * 64];
        }
        finish(i, b, v);
      }
    }
  }
  return F16 || __ballot(odd != 0.f) == 0;
}

template <int WM, int WN, int NB, int KW, int TM>
__global__ __launch_bounds__(64 * WM * WN * KW, NB == 1 ? 3 : 2) void half_kernel(const MatArguments) {
  Arguments arguments = (Arguments)__builtin_amdgcn_kernarg_segment_ptr();
  const int id = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (id >= arguments->g.ptiles * arguments->g.mtiles * arguments->g.csplit) return;
  if (matrix_pass<0, WM, WN, NB, KW, TM>(arguments, threadIdx.x)) return;
  int thread = threadIdx.x;
  asm("" : "+s"(arguments), "+v"(thread));  // so that nothing that a pass computed is kept for the next
  if (matrix_pass<1, WM, WN, NB, KW, TM>(arguments, thread)) return;
  asm("" : "+s"(arguments), "+v"(thread));
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the last pass stores over what the second has stored, by other lanes
  matrix_pass<2, WM, WN, NB, KW, TM>(arguments, thread);
}

// ---- the weights, made once per filter and chunk size ---------------------------------------------------------------------
// packed streams -> the dense filter, channels innermost (`cpad` of them); one wave per stream
__global__ __launch_bounds__(256) void dense_kernel(const int32_t* __restrict__ grp_off, const int32_t* __restrict__ grp_nnz,
                                                    const int32_t* __restrict__ oc_order, const int32_t* __restrict__ position,
                                                    const float* __restrict__ values, float* __restrict__ dense, int C, int K, int ks,
                                                    int tile_ic, int stages, int G, int nstream, int cpad) {
  const int sid = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (sid >= nstream) return;
  const int grp = sid / stages, st = sid - grp * stages;
  const int beg = grp_off[sid], n = grp_nnz[sid];
  for (int i = lane; i < n; i += 64) {
    const unsigned pos = (unsigned)position[beg + i];
    const int s = pos & 7, r = (pos >> 3) & 7, ic = st * tile_ic + (int)((pos >> 6) & 0x3ffff);
    const int oc = oc_order[grp * G + (int)(pos >> 24)];
    if (oc < 0 || oc >= K || ic >= C) continue;
    dense[(((size_t)oc * ks + r) * ks + s) * cpad + ic] = values[beg + i];
  }
}

// What making a plan writes.
struct MatLists {
  int* wide;      // not zero: some weight is not the sum of its parts
  int* count;     // steps of every (32 output channels, chunk)
  int* first;     // the sums before them, and of them all
  int* row_exp;
  int* loose_count;
  int2* loose;
  char* steps;
  char* slots;
};
constexpr int kMostCounts = 2048;  // of a plan whose workgroups each add up the counts before their own

// A workgroup per 32 output channels and chunk of 8*kgs input channels.  The chunk's blocks -- one tap of 8 channels -- are put
// four to a step; a block with three or four weights in a group of four channels comes twice, the second time with the
// third and the fourth.  Blocks of zeros are left out.
// FILL false: counts the steps only; the workgroups beyond those find the exponents of the rows' largest weights, a wave per row.
// Latency of a workgroup's few rounds bounds both, so 1024 threads: 6 and 16 us on average over four layers, with 256 8 and 18.
template <bool FILL>
__global__ __launch_bounds__(1024) void steps_kernel(const MatWeights w, const MatLists out, int K, int ks, int kgs, int chunks, int mblocks) {
  constexpr int kMost = 256, kThreads = 1024;
  __shared__ int layers[kMost];
  __shared__ int list[2 * kMost];
  __shared__ int listed;
  __shared__ int before[kThreads / 64];
  const int id = blockIdx.x, counts = chunks * mblocks, block = id / chunks, chunk = id - block * chunks, taps = ks * ks, subs = kgs * taps;
  if (!FILL && id >= counts) {
    const int row = (id - counts) * (kThreads / 64) + threadIdx.x / 64, per_row = taps * chunks * 8 * kgs;
    if (row >= 32 * mblocks) return;
    float most = 0;
    if (row < K) {
      const float4* values = reinterpret_cast<const float4*>(w.dense + (size_t)row * per_row);
#pragma unroll 4
      for (int i = threadIdx.x & 63; i < per_row / 4; i += 64) {
        const float4 f = values[i];
        most = fmaxf(fmaxf(fmaxf(most, fabsf(f.x)), fmaxf(fabsf(f.y), fabsf(f.z))), fabsf(f.w));
      }
    }
    for (int d = 32; d; d >>= 1) most = fmaxf(most, __shfl_xor(most, d));
    if ((threadIdx.x & 63) == 0) out.row_exp[row] = most > 0 ? ilogbf(most) - 14 : 0;
    return;
  }
  auto weights = [&](int row, int sub, int group) {  // four channels of a block
    const int oc = block * 32 + row, tap = sub / kgs;
    const float4* d = reinterpret_cast<const float4*>(w.dense + (((size_t)oc * taps + tap) * chunks + chunk) * 8 * kgs);
    return oc < K ? d[2 * (sub - tap * kgs) + group] : make_float4(0.f, 0.f, 0.f, 0.f);
  };
  for (int i = threadIdx.x; i < subs; i += kThreads) layers[i] = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < subs * 64; i += kThreads) {
    const int sub = i >> 6, row = i & 31, group = i >> 5 & 1;
    const float4 f = weights(row, sub, group);
    const int n = (f.x != 0.f) + (f.y != 0.f) + (f.z != 0.f) + (f.w != 0.f);
    if (n) atomicMax(&layers[sub], (n + 1) / 2);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int n = 0;
    for (int layer = 0; layer < 2; ++layer)
      for (int sub = 0; sub < subs; ++sub)
        if (layers[sub] > layer) list[n++] = sub | layer << 16;
    listed = n;
    if (!FILL) out.count[id] = max(1, (n + 3) / 4);
  }
  if (!FILL) return;
  // the steps before these: summed here, or where they are many by first_kernel
  int first = 0;
  if (counts <= kMostCounts) {
    for (int i = threadIdx.x; i < id; i += kThreads) first += out.count[i];
    for (int d = 32; d; d >>= 1) first += __shfl_xor(first, d);
    if ((threadIdx.x & 63) == 0) before[threadIdx.x / 64] = first;
  }
  __syncthreads();
  const int n = listed, steps_here = max(1, (n + 3) / 4), items = steps_here * 64;
  if (counts <= kMostCounts) {
    first = 0;
    for (int i = 0; i < kThreads / 64; ++i) first += before[i];
    if (threadIdx.x == 0) out.first[id] = first;
    if (threadIdx.x == 0 && id == counts - 1) out.first[counts] = first + steps_here;
  } else {
    first = out.first[id];
  }
  if (id == counts - 1 && threadIdx.x < 192)  // what is read ahead of the end names a block that exists
    *reinterpret_cast<unsigned*>(out.steps + (size_t)(first + steps_here + (int)threadIdx.x / 64) * kStepBytes + 3072 + threadIdx.x % 64 * 4) = 0;
  for (int i = threadIdx.x; i < items; i += kThreads) {
    const int step = i >> 6, lane = i & 63, row = lane & 31, half = lane >> 5;
    // eight slots: blocks 2 half and 2 half + 1 of the step, two groups of four channels each, two slots a group
    unsigned index = 0;
    const int shift = -w.row_exp[block * 32 + row];
    float v[8], scaled[8];
    for (int k = 0; k < 4; ++k) {
      const int at = 4 * step + 2 * half + k / 2, entry = at < n ? list[at] : -1;
      int found = 0, place[2] = {0, 3};
      float value[2] = {0, 0};
      const int sub = entry & 0xffff;
      if (entry >= 0) {
        const float4 four = weights(row, sub, k & 1);
        for (int j = 0; j < 4; ++j) {
          const float f = j == 0 ? four.x : j == 1 ? four.y : j == 2 ? four.z : four.w;
          if (f == 0.f) continue;
          const int slot = found++ - 2 * (entry >> 16);
          if (slot == 0 || slot == 1) {
            place[slot] = j;
            value[slot] = f;
          }
        }
      }
      if (place[0] == 3) {  // the two places of a group ascend
        place[0] = 0; place[1] = 3;
        value[1] = value[0]; value[0] = 0;
      }
      index |= (unsigned)(place[0] | place[1] << 2) << (4 * k);
      for (int slot = 0; slot < 2; ++slot) {
        v[2 * k + slot] = value[slot];
        scaled[2 * k + slot] = ldexpf(value[slot], shift);
        if (value[slot] == 0.f || fabsf(scaled[2 * k + slot]) >= kLeast) continue;
        const int tap = sub / kgs, n = atomicAdd(out.loose_count + block, 1);
        if (n >= kMostLoose || !(fabsf(scaled[2 * k + slot]) >= kLeastLoose)) *out.wide = 1;
        else out.loose[kMostLoose * block + n] = make_int2(row | tap / ks << 5 | tap % ks << 8 |
                                                           ((chunk * kgs + sub - tap * kgs) * 8 + 4 * (k & 1) + place[slot]) << 11,
                                                       (int)bits_of(scaled[2 * k + slot]));
        scaled[2 * k + slot] = 0;
      }
    }
    // the blocks that this lane reads the input of: one in each half of its registers
    unsigned code[2];
    for (int r = 0; r < 2; ++r) {
      const int at = 4 * step + 2 * r + half, sub = at < n ? list[at] & 0xffff : 0, tap = sub / kgs, kg = sub - tap * kgs;
      const int bits = ks > 4 ? 3 : 2;  // seven bits: column and row of the tap, channel group
      code[r] = (unsigned)(tap % ks | tap / ks << bits | kg << 2 * bits);
    }
    const size_t to = first + step;
    char* dst = out.steps + to * kStepBytes;
    *reinterpret_cast<unsigned*>(dst + 3072 + lane * 4) = index | code[0] << 16 | code[1] << 24 | (step + 1 == steps_here ? 0x80000000u : 0u);
    u32x4 h, m, l;
    unsigned rest = 0;
    f16x2 zeros = {0, 0};
    cut16(scaled, 1.f, h, m, l, zeros, &rest);
    if (rest) *out.wide = 1;
    l = __builtin_bit_cast(u32x4, __builtin_bit_cast(f16x8, l) * (f16x8)(_Float16)(1 / kLow));
    *reinterpret_cast<u32x4*>(dst + lane * 16) = h;
    *reinterpret_cast<u32x4*>(dst + 1024 + lane * 16) = m;
    *reinterpret_cast<u32x4*>(dst + 2048 + lane * 16) = l;
    char* raw = out.slots + to * kSlotBytes + lane * 16;
    *reinterpret_cast<u32x4*>(raw) = u32x4{bits_of(v[0]), bits_of(v[1]), bits_of(v[2]), bits_of(v[3])};
    *reinterpret_cast<u32x4*>(raw + 1024) = u32x4{bits_of(v[4]), bits_of(v[5]), bits_of(v[6]), bits_of(v[7])};
  }
}

// Puts a block's loose weights in order, so that sums do not depend on who came first; their count is -1 where the first pass cannot
// be made.
__global__ __launch_bounds__(64) void loose_kernel(const int* __restrict__ wide, int* __restrict__ loose_count, int2* __restrict__ loose) {
  if (*wide) {
    if (threadIdx.x == 0) loose_count[blockIdx.x] = -1;
    return;
  }
  __shared__ int2 list[kMostLoose];
  const int n = min(loose_count[blockIdx.x], kMostLoose), i = threadIdx.x;
  int2* all = loose + kMostLoose * blockIdx.x;
  if (i < n) list[i] = all[i];
  __syncthreads();
  if (i >= n) return;
  int before = 0;
  for (int k = 0; k < n; ++k) before += list[k].x < list[i].x;
  all[before] = list[i];
}

// counts -> the first step of every (32 output channels, chunk)
__global__ __launch_bounds__(1024) void first_kernel(const int* __restrict__ count, int* __restrict__ first, int n) {
  __shared__ int sums[1024];
  int before = 0;
  for (int at = 0; at < n; at += 1024) {
    const int i = at + (int)threadIdx.x, mine = i < n ? count[i] : 0;
    sums[threadIdx.x] = mine;
    __syncthreads();
    for (int d = 1; d < 1024; d <<= 1) {
      const int v = (int)threadIdx.x >= d ? sums[threadIdx.x - d] : 0;
      __syncthreads();
      sums[threadIdx.x] += v;
      __syncthreads();
    }
    if (i < n) first[i] = before + sums[threadIdx.x] - mine;
    before += sums[1023];
    __syncthreads();
  }
  if (threadIdx.x == 0) first[n] = before;
}

template <int WM, int WN, int NB, int KW, int TM>
int launch_one(const MatGeom& g, const float* d_in, float* d_out, const MatWeights& weights, hipStream_t stream) {
  auto kern = half_kernel<WM, WN, NB, KW, TM>;
  static std::atomic<bool> lds_set{false};  // per instantiation; setting the attribute twice is harmless
  if (!lds_set.load(std::memory_order_acquire)) {
    TETRIS_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kMatLds));
    lds_set.store(true, std::memory_order_release);
  }
  const int grid = 8 * ceil_div(g.ptiles * g.mtiles * g.csplit, 8);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * WM * WN * KW), mat_lds_bytes(g), stream, MatArguments{d_in, d_out, weights, g});
  TETRIS_HIP(hipGetLastError());
  return TETRIS_OK;
}

size_t dense_bytes(const MatGeom& g) { return (size_t)g.K * g.ks * g.ks * g.chunks * 8 * g.kgs * sizeof(float); }

// one allocation: first what has to be zero (flag, counts of loose weights, dense filter), then the rows' exponents, the steps' counts
// and sums, the loose weights, the steps, their weights as they are
MatWeights mat_weights_at(const MatGeom& g, void* base, size_t* bytes, size_t* zeros = nullptr, MatLists* lists = nullptr) {
  size_t at = 0;
  auto take = [&](size_t n) {
    char* p = static_cast<char*>(base) + at;
    at += (n + 255) / 256 * 256;
    return p;
  };
  const size_t steps = (size_t)g.mblocks * g.chunks * g.smax + 3;  // (waves read ahead)
  MatLists l{};
  l.wide = reinterpret_cast<int*>(take(sizeof(int)));
  l.loose_count = reinterpret_cast<int*>(take((size_t)g.mblocks * 4));
  MatWeights w{};
  w.base = base;
  w.dense = reinterpret_cast<const float*>(take(dense_bytes(g)));
  if (zeros) *zeros = at;
  l.row_exp = reinterpret_cast<int*>(take((size_t)g.mblocks * 32 * 4));
  l.count = reinterpret_cast<int*>(take((size_t)g.mblocks * g.chunks * 4));
  l.first = reinterpret_cast<int*>(take(((size_t)g.mblocks * g.chunks + 1) * 4));
  l.loose = reinterpret_cast<int2*>(take((size_t)g.mblocks * kMostLoose * 8));
  l.steps = take(steps * kStepBytes);
  l.slots = take(steps * kSlotBytes);
  w.row_exp = l.row_exp;
  w.first = l.first;
  w.loose_count = l.loose_count;
  w.loose = l.loose;
  w.steps = l.steps;
  w.slots = l.slots;
  w.step_bytes = (int)(steps * kStepBytes);
  if (bytes) *bytes = at;
  if (lists) *lists = l;
  return w;
}

}  // namespace

size_t half_weight_bytes(const MatGeom& g) {
  size_t bytes = 0;
  mat_weights_at(g, nullptr, &bytes);
  return bytes;
}

int half_weights(const tetris_g950* p, const MatGeom& g, hipStream_t stream, void* base, MatWeights* out) {
  MatLists l;
  size_t zeros = 0;
  const MatWeights w = mat_weights_at(g, base, nullptr, &zeros, &l);
  TETRIS_HIP(hipMemsetAsync(base, 0, zeros, stream));
  const int nstream = p->groups * p->stages, counts = g.chunks * g.mblocks;
  hipLaunchKernelGGL(dense_kernel, dim3(ceil_div(nstream, 4)), dim3(256), 0, stream, p->d_grp_off, p->d_grp_nnz, p->d_oc_order,
                     p->d_position, p->d_values, const_cast<float*>(w.dense), p->C, p->K, p->ks, p->tile_ic, p->stages, p->g, nstream,
                     8 * g.kgs * g.chunks);
  hipLaunchKernelGGL(steps_kernel<false>, dim3(counts + 2 * g.mblocks), dim3(1024), 0, stream, w, l, g.K, g.ks, g.kgs, g.chunks, g.mblocks);
  if (counts > kMostCounts) hipLaunchKernelGGL(first_kernel, dim3(1), dim3(1024), 0, stream, l.count, l.first, counts);
  hipLaunchKernelGGL(steps_kernel<true>, dim3(counts), dim3(1024), 0, stream, w, l, g.K, g.ks, g.kgs, g.chunks, g.mblocks);
  hipLaunchKernelGGL(loose_kernel, dim3(g.mblocks), dim3(64), 0, stream, l.wide, l.loose_count, l.loose);
  TETRIS_HIP(hipGetLastError());
  // launches on other streams may follow at once
  TETRIS_HIP(hipStreamSynchronize(stream));
  *out = w;
  return TETRIS_OK;
}

int launch_half(const MatGeom& g, const float* d_in, float* d_out, const MatWeights& weights, int relu, hipStream_t stream) {
  MatGeom k = g;
  k.relu = relu;
  k.quads = stores_quads(g, d_out);
  const MatShape& c = kMatShapes[g.cfg];
  const bool two = g.kgs * g.lpad / 64 <= 2 * c.wm * c.wn;
#define TETRIS_MAT(WM, WN, NB, KW) \
  if (c.wm == WM && c.wn == WN && c.nb == NB && c.kw == KW) \
    return two ? launch_one<WM, WN, NB, KW, 2>(k, d_in, d_out, weights, stream) \
               : launch_one<WM, WN, NB, KW, NB == 4 ? 2 : kMatTasks>(k, d_in, d_out, weights, stream);
  TETRIS_MAT(8, 1, 2, 1) TETRIS_MAT(4, 1, 2, 2) TETRIS_MAT(2, 2, 1, 1) TETRIS_MAT(2, 2, 1, 2) TETRIS_MAT(8, 1, 3, 1) TETRIS_MAT(4, 2, 3, 1) TETRIS_MAT(8, 1, 4, 1)
  TETRIS_MAT(4, 2, 4, 1)
#undef TETRIS_MAT
  return fail(TETRIS_EINVAL, "no matrix kernel of configuration %d", g.cfg);
}

}  // namespace tetris
