// What the two matrix kernels (matrix_conv.hip, matrix_half.hip) share.
#pragma once
#include "common.h"

namespace tetris {

// A workgroup of a configuration: waves along the channels and along the pixels of a team, pixel blocks of a wave, teams;
// whether half_kernel runs it, and with short chunks of channels.  (half_kernel's: those that are left if of 22 and four more the
// ones are dropped one after the other that the 424 layers of profiles/kernel_times.txt lose least without, 0.01 % in all.)
struct MatShape {
  int wm, wn, nb, kw;
  bool half, brief;
};
constexpr MatShape kMatShapes[] = {
    {4, 1, 4, 1}, {4, 1, 4, 2}, {4, 1, 2, 1}, {4, 1, 2, 2}, {4, 1, 2, 4}, {2, 2, 2, 1}, {2, 2, 2, 2}, {2, 2, 2, 4}, {2, 2, 1, 1}, {2, 2, 1, 2}, {2, 2, 1, 4},
    {8, 1, 2, 1, true}, {8, 1, 3, 1, true}, {4, 1, 2, 2, true}, {2, 2, 1, 2, true},
    {8, 1, 2, 1, true, true}, {8, 1, 3, 1, true, true}, {8, 1, 4, 1, true, true}, {4, 2, 3, 1, true, true}, {4, 2, 4, 1, true, true},
    {4, 1, 2, 2, true, true}, {2, 2, 1, 1, true, true}, {2, 2, 1, 2, true, true}};
static_assert(sizeof kMatShapes / sizeof *kMatShapes == kMatConfigs);

// whether four consecutive pixels of a tile lie side by side in memory, in one image and on 16 bytes
inline bool stores_quads(const MatGeom& g, const float* d_out) {
  return !g.pool && g.strips == 1 && g.OH * g.OW % 4 == 0 && reinterpret_cast<uintptr_t>(d_out) % 16 == 0;
}

// matrix_half.hip
constexpr int kMostChannels = 1 << 20;  // input channels of a layer: a loose weight's place is an int, 20 bits of which name its channel
constexpr int kAsideBytes = 64 + 64 * 8;  // of LDS: inputs that are multiplied one by one
constexpr int kStepBytes = 3 * 1024 + 256, kSlotBytes = 2048;  // of a step's weights: fp16 parts and a word per lane; fp32
size_t half_weight_bytes(const MatGeom& g);
int half_weights(const tetris_g950* p, const MatGeom& g, hipStream_t stream, void* base, MatWeights* out);  // waits for them
int launch_half(const MatGeom& g, const float* d_in, float* d_out, const MatWeights& weights, int relu, hipStream_t stream);

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int kOutside = 0x7ff00000;  // a byte offset beyond every tensor this path takes (1 GiB): loads give 0, stores are dropped

constexpr float kScale = 0x1p32f, kUnscale = 0x1p-64f;  // bf16 parts: inputs and weights times 2^32, sums times 2^-64

// three bf16 parts of eight floats, scaled
__device__ __forceinline__ void cut(const float (&x)[8], u32x4& hi, u32x4& mid, u32x4& lo) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x2 v = {x[2 * i] * kScale, x[2 * i + 1] * kScale};
    const unsigned h = __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
    const float r0 = v.x - __builtin_bit_cast(float, h << 16), r1 = v.y - __builtin_bit_cast(float, h & 0xffff0000u);
    const unsigned m = __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{r0, r1}, bf16x2));
    const float s0 = r0 - __builtin_bit_cast(float, m << 16), s1 = r1 - __builtin_bit_cast(float, m & 0xffff0000u);
    hi[i] = h;
    mid[i] = m;
    lo[i] = __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{s0, s1}, bf16x2));
  }
}

__device__ __forceinline__ unsigned bits_of(float x) { return __builtin_bit_cast(unsigned, x); }

// maximum over the four lanes of a quad
__device__ __forceinline__ float quad_max(float v) {
  v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xf, 0xf, true)));
  return fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xf, 0xf, true)));
}

// value k of lane q of four neighbours becomes value q of lane k
__device__ __forceinline__ void transpose_quad(float (&v)[4], int lane) {
  auto from = [](float x, auto lanes) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(lanes)::value, 0xf, 0xf, true));
  };
  constexpr std::integral_constant<int, 0xB1> beside;  // lane ^ 1
  constexpr std::integral_constant<int, 0x4E> across;  // lane ^ 2
  const bool odd = lane & 1, high = lane & 2;
  float o[4], a[4];  // (the exchanges outside of the choices: all lanes take part)
#pragma unroll
  for (int k = 0; k < 4; ++k) o[k] = from(v[k ^ 1], beside);
#pragma unroll
  for (int k = 0; k < 4; ++k) a[k] = odd == (k & 1) ? v[k] : o[k];
#pragma unroll
  for (int k = 0; k < 4; ++k) o[k] = from(a[k ^ 2], across);
#pragma unroll
  for (int k = 0; k < 4; ++k) v[k] = high == (k >> 1) ? a[k] : o[k];
}

}  // namespace
}  // namespace tetris
