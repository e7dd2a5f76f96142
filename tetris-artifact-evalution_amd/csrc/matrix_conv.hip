// Convolution of a sparse filter as a dense product on the matrix cores, for layers whose filter is not sparse enough, or
// whose launch is not large enough, for the kernels that walk the non-zeros (spconv2d_kernel.hip).
//
// A vector FMA with a scalar weight does 16 multiply-adds a cycle and SIMD and the walk reaches two thirds of that, on the
// non-zeros only.  The matrix cores do 512 a cycle and SIMD in bf16.  An fp32 number is the sum of three bf16 numbers,
// exactly (8 + 8 + 8 bits of significand, each part rounded to nearest: the second is at most 2^-8 of the first, the
// third 2^-17), and of the nine products of two such sums all but the last, low times low, are formed here: that one is
// 2^-34 of the product at most.  (Without mid times low and low times mid, up to 2^-25 each, an output of one term was
// off by up to 8.6e-8 of itself where one rounding to fp32 is off by 6.0e-8.)  Sums stay in fp32.  That is 64 fp32
// multiply-adds a cycle and SIMD on ALL weights, zeros included.  (Parts in bf16: Henry, Tang and Heinecke, "Leveraging the
// bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations", ARITH 2019.)
//
// Workgroup: KW teams of four waves on one tile of 32*WM output channels x P = 32*NB*(4/WM) output pixels.  The input of P
// pixels (with its halo) of 8*kgs channels at a time is read from the NCHW image, cut into its three parts once, and
// kept in LDS as [channel group of 8][part][pixel][8 channels]: a lane's eight k-values of a product are one aligned
// 16-byte read, the lanes of a row read consecutive addresses, and another kernel tap is another constant offset, so
// the parts are made once for all ks*ks taps.  Weights were cut when the plan was made and lie in the order the lanes load
// them (1 KiB per 32 channels, 16 k-values and part): they go from L2 to registers, past LDS, because the four waves along
// the channels share none.  The teams take the chunks of channels in turn and add their sums in LDS at the end: four waves
// on every SIMD also where a layer has one tile per CU (16 x 128 x 28 x 28, 3x3: 36 us with one team, 31 with two).
//
// What bounds it: on large layers the matrix cores (128 -> 256 channels, 52x52, batch 16: 148 us, 1.38 PFLOP/s of bf16
// products, where the vendor's bf16 GEMM of 8192^3 reaches 1.37); on small ones the latency of a round: weights from L2,
// input from HBM, barrier.
//
// Range: parts are made of numbers scaled by 2^32, inputs and weights, so that the lowest bit of every fp32 number, subnormal
// ones too, is a normal bf16 number's, and sums are scaled back as they are stored.  What is out of that range upwards
// (an infinity, NaN, an input of 2^96 or more, a sum of 2^64 or more) makes every sum that it enters infinite or NaN,
// whatever the weight: a wave that finds such a sum computes its outputs once more as the walking kernels do, with FMAs on
// the non-zero weights only.  Packs with weights of 2^64 or more, or not finite, stay with those kernels.
#include <algorithm>
#include <cmath>
#include <numeric>

#include "matrix.h"

namespace tetris {
namespace {

__device__ __forceinline__ f32x16 product(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// x / d for x below 2^30
__device__ __forceinline__ int quotient(int x, MatDiv d) { return (int)((unsigned long long)(unsigned)x * d.m >> d.shift); }

template <int WM, int NB, int KW, int TM>
__global__ __launch_bounds__(256 * KW, KW == 4 ? 4 : 2) void matrix_kernel(const float* __restrict__ in, float* __restrict__ out,
                                                        const u32x4* __restrict__ weights, const MatGeom g) {
  constexpr int WN = 4 / WM, P = 32 * NB * WN;
  extern __shared__ u32x4 all_lds[];  // [KW][2][kgs][3][lpad]
  const int lane = threadIdx.x & 63, team = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8),
            wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3);
  u32x4* const lds = all_lds + team * 6 * g.kgs * g.lpad;
  // workgroup ids go round-robin to the XCDs: each XCD gets a contiguous range of logical ids.  Channel blocks of one pixel
  // tile are neighbours (they read the same input), slices outermost (they share nothing).
  const int per = gridDim.x >> 3;
  const int id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  const int tiles = g.ptiles * g.mtiles;
  if (id >= tiles * g.csplit) return;
  const int slice = quotient(id, g.d_tiles), tile = id - slice * tiles;
  const int pt = quotient(tile, g.d_mtiles), mt = tile - pt * g.mtiles;
  const int wm = wave % WM, wn = wave / WM;

  // first pixel of the tile: strip image q0, row and column in it (in 2x2 blocks when pooling)
  const int psh = g.pool ? 2 : 0, dbl = g.pool ? 1 : 0;
  const int u0 = (pt * P) >> psh;
  const int q0 = quotient(u0, g.d_upq), r0 = u0 - q0 * g.upq;
  const int oy0 = quotient(r0, g.d_uw), ox0 = r0 - oy0 * g.uw;
  const int row0 = (oy0 << dbl) * g.stride, col0 = (ox0 << dbl) * g.stride;

  // the teams of a workgroup take the slice's chunks in turn
  const int c_beg = slice * g.chunks / g.csplit + team, c_end = (slice + 1) * g.chunks / g.csplit;
  const int rounds = (c_end - c_beg + team + KW - 1) / KW;
  const int halves = g.kgs >> 1, per_chunk = g.ks * g.ks * halves;
  const u32x4* wp = weights + (size_t)min(mt * WM + wm, g.mblocks - 1) * g.steps * 192 + lane;
  u32x4 a[3];
  auto fetch_weights = [&](int step) {
#pragma unroll
    for (int p = 0; p < 3; ++p) a[p] = wp[(size_t)step * 192 + p * 64];
  };

  // The first weights and the first input are asked for before anything that they do not depend on is computed.
  if (c_beg < c_end) fetch_weights(c_beg * per_chunk);

  // what this wave stages: 64 staged pixels of one channel group per task
  const int blocks = g.lpad >> 6, tasks = g.kgs * blocks;
  int goff[TM], gkg[TM], gslot[TM];
#pragma unroll
  for (int k = 0; k < TM; ++k) {
    const int task = wave + 4 * k;
    gkg[k] = quotient(task, g.d_blocks);
    const int blk = task - gkg[k] * blocks;
    gslot[k] = gkg[k] * 3 * g.lpad + blk * 64 + lane;
    const unsigned x = col0 + blk * 64 + lane;
    const unsigned dr = g.wp == 1 ? x : __umulhi(x, g.m_wp), col = x - dr * g.wp;
    const unsigned row = row0 + dr;
    const unsigned dq = g.ihs == 1 ? row : __umulhi(row, g.m_ihs), y = row - dq * g.ihs;
    const unsigned q = q0 + dq, n = g.strips == 1 ? q : __umulhi(q, g.m_strips), strip = q - n * g.strips;
    const int iy = (int)y * g.sub - g.pad, ix = (int)(strip * g.ws * g.stride + col) * g.sub - g.pad;
    goff[k] = task < tasks && n < (unsigned)g.N && iy >= 0 && iy < g.H && ix >= 0 && ix < g.W
                  ? 4 * (int)(n * (unsigned)(g.C * g.H * g.W) + (unsigned)(iy * g.W + ix)) : kOutside;
  }
  const int hw4 = 4 * g.H * g.W;
  const __amdgpu_buffer_rsrc_t irsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(in), 0, g.in_bytes, 0x00020000);
  float x[TM][8];
  auto fetch = [&](int chunk) {
#pragma unroll
    for (int k = 0; k < TM; ++k) {
      if (wave + 4 * k >= tasks) break;
      const int c = (chunk * g.kgs + gkg[k]) * 8;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        x[k][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                irsrc, c + j < g.C ? goff[k] : kOutside, min(c + j, g.C - 1) * hw4, 0));
    }
  };
  auto keep = [&](int buf) {
#pragma unroll
    for (int k = 0; k < TM; ++k) {
      if (wave + 4 * k >= tasks) break;
      u32x4 h, m, l;
      cut(x[k], h, m, l);
      u32x4* d = lds + buf * 3 * g.kgs * g.lpad + gslot[k];
      d[0] = h;
      d[g.lpad] = m;
      d[2 * g.lpad] = l;
    }
  };

  if (c_beg < c_end) fetch(c_beg);

  // where this lane's pixels lie: in the output's images, in LDS and in the output
  struct Pixel { bool in_range; int t; unsigned n, dq, uy, oy, ox, w; };  // ox: in its strip, w: in its image
  auto pixel = [&](int b, int lane) {
    Pixel p;
    const int t = (wn * NB + b) * 32 + (lane & 31);
    p.in_range = pt * P + t < g.npix;
    p.t = p.in_range ? t : g.npix - 1 - pt * P;
    const unsigned x = ox0 + (p.t >> psh);
    const unsigned dy = __umulhi(x, g.m_uw), ux = g.uw == 1 ? 0 : x - dy * g.uw;
    const unsigned y = oy0 + (g.uw == 1 ? x : dy);
    p.dq = g.uh == 1 ? y : __umulhi(y, g.m_uh);
    p.uy = y - p.dq * g.uh;
    p.oy = (p.uy << dbl) + (g.pool ? (p.t >> 1) & 1 : 0);
    p.ox = (ux << dbl) + (g.pool ? p.t & 1 : 0);
    const unsigned q = q0 + p.dq;
    p.n = g.strips == 1 ? q : __umulhi(q, g.m_strips);
    p.w = (q - p.n * g.strips) * g.ws + p.ox;
    return p;
  };
  int bpos[NB], ooff[NB];
  const int ohw = g.pool ? (g.OH >> 1) * (g.OW >> 1) : g.OH * g.OW;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const Pixel p = pixel(b, lane);
    bpos[b] = ((int)(p.dq * g.ihs + p.oy * g.stride) - row0) * g.wp + (int)p.ox * g.stride - col0 + (lane >> 5) * 3 * g.lpad;
    if (g.pool)
      ooff[b] = p.in_range && (p.t & 3) == 0 && (p.w >> 1) < (unsigned)(g.OW >> 1)
                    ? 4 * (int)((p.n * g.K + 4 * (lane >> 5)) * ohw + p.uy * (g.OW >> 1) + (p.w >> 1)) : kOutside;
    else
      ooff[b] = p.in_range && p.w < (unsigned)g.OW ? 4 * (int)((p.n * g.K + 4 * (lane >> 5)) * ohw + p.oy * g.OW + p.w) : kOutside;
  }

  // The products of the leading parts and the seven small ones are summed apart: a sum of its own is rounded once per 16
  // k-values, not eight times, and the small ones are 2^-8 of it.
  f32x16 acc[NB], low[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[b][i] = low[b][i] = 0.f;
  if (c_beg < c_end) keep(0);
  __syncthreads();
  int buf = 0;
  for (int round = 0; round < rounds; ++round) {
    const int chunk = c_beg + round * KW;
    if (chunk < c_end) {
      const bool more = chunk + KW < c_end;
      const u32x4* tile_lds = lds + buf * 3 * g.kgs * g.lpad;
      int r = 0, s = 0, half = 0;
      for (int i = 0; i < per_chunk; ++i) {
        const u32x4* src = tile_lds + r * g.wp + s + half * 6 * g.lpad;
        // The next step's weights are asked for ahead of this step's products -- with four teams, whose registers do not hold
        // two steps, behind them: the other teams' products fill the wait --, the next chunk's input behind the second
        // step's weights, so that these do not wait for it.
        u32x4 w[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) w[p] = a[p];
        auto ahead = [&]() {
          if (i + 1 < per_chunk) fetch_weights(chunk * per_chunk + i + 1);
          else if (more) fetch_weights((chunk + KW) * per_chunk);
          if (i == 0 && more) fetch(chunk + KW);
        };
        if constexpr (KW < 4) ahead();
        if (++half == halves) {
          half = 0;
          if (++s == g.ks) { s = 0; ++r; }
        }
        // the eight products, smallest first
        constexpr int pa[8] = {2, 1, 2, 1, 0, 1, 0, 0}, pb[8] = {1, 2, 0, 1, 2, 0, 1, 0};
        if constexpr (KW < 4) {
          u32x4 v[NB][3];
#pragma unroll
          for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int p = 0; p < 3; ++p) v[b][p] = src[bpos[b] + p * g.lpad];
#pragma unroll
          for (int t = 0; t < 8; ++t)
#pragma unroll
            for (int b = 0; b < NB; ++b) {
              f32x16& sum = t == 7 ? acc[b] : low[b];
              sum = product(w[pa[t]], v[b][pb[t]], sum);
            }
        } else {
#pragma unroll
          for (int b = 0; b < NB; ++b) {
            u32x4 v[3];
#pragma unroll
            for (int p = 0; p < 3; ++p) v[p] = src[bpos[b] + p * g.lpad];
#pragma unroll
            for (int t = 0; t < 8; ++t) {
              f32x16& sum = t == 7 ? acc[b] : low[b];
              sum = product(w[pa[t]], v[pb[t]], sum);
            }
          }
          ahead();
        }
      }
      if (more) keep(buf ^ 1);
    }
    buf ^= 1;
    __syncthreads();
  }

  float* dst = out + (size_t)slice * g.out_floats;
  const __amdgpu_buffer_rsrc_t orsrc = __builtin_amdgcn_make_buffer_rsrc(dst, 0, 4 * g.out_floats, 0x00020000);
  const int oc0 = (mt * WM + wm) * 32;
  // sum i of a lane: channel 8*(i/4) + 4*(lane/32) + i%4 of its wave's 32, pixel lane%32
  auto store = [&](int i, int b, float v) {
    const int oc = oc0 + 8 * (i / 4) + i % 4;
    if (g.pool) v = quad_max(v);
    if (g.relu) v = fmaxf(v, 0.f);
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, v), orsrc, oc + 4 * (lane >> 5) < g.K ? ooff[b] : kOutside, oc * ohw * 4, 0);
  };
  float odd = 0;  // NaN once a sum is infinite or NaN
  auto finish = [&](int i, int b, float (&v)[4]) {  // sums i to i + 3
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      odd = fmaf(v[k], 0.f, odd);
      v[k] *= kUnscale;
    }
    if (g.quads) {
      // Four pixels of a channel to a lane instead of four channels of a pixel: a store of 16 bytes instead of four.  The
      // stores, 16 cycles each for the address unit of a CU, are what the end of a tile waits for.
      transpose_quad(v, lane);
      u32x4 d;
#pragma unroll
      for (int k = 0; k < 4; ++k) d[k] = bits_of(g.relu ? fmaxf(v[k], 0.f) : v[k]);
      const bool inside = oc0 + 2 * i + 4 * (lane >> 5) + (lane & 3) < g.K && ooff[b] != kOutside;
      __builtin_amdgcn_raw_buffer_store_b128(d, orsrc, inside ? ooff[b] + 4 * (lane & 3) * (ohw - 1) : kOutside, (oc0 + 2 * i) * ohw * 4, 0);
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
        float v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = acc[b][i + k] + low[b][i + k];
        finish(i, b, v);
      }
  } else {
    // every team leaves its sums in LDS and adds a share of all of them
    float* sums = reinterpret_cast<float*>(all_lds) + wave * 1024 * NB + lane;
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
      for (int b = 0; b < NB; ++b) sums[team * 4096 * NB + (i * NB + b) * 64] = acc[b][i] + low[b][i];
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
          for (int k = 1; k < KW; ++k) v[j] += sums[k * 4096 * NB + ((i + j) * NB + b) * 64];
        }
        finish(i, b, v);
      }
    }
  }
  if (__ballot(odd != 0.f) == 0) return;
  // Out of range: the wave's sums once more, over what was stored.  (Not always by the same lane: where outputs went out four pixels
  // at a time an output's lane was its neighbour.  So the wave waits until they are there.)
  // Latency of the loads bounds this, and it is here to be right: 1.7 ms with one infinity in the input of the layer above
  // (128 -> 256 channels, 52x52, batch 16), 3.9 ms with nothing but.
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  int again = lane;  // (unknown to the compiler, which would else keep the pixels' places in registers all the while)
  asm("" : "+v"(again));
  const int ch0 = slice * g.chunks / g.csplit * 8 * g.kgs, ch1 = min(g.C, (slice + 1) * g.chunks / g.csplit * 8 * g.kgs);
  const u32x4* block = weights + (size_t)min(mt * WM + wm, g.mblocks - 1) * g.steps * 192;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const Pixel p = pixel(b, again);
    float sum[16 / KW];
#pragma unroll
    for (int j = 0; j < 16 / KW; ++j) sum[j] = 0;
#pragma nounroll
    for (int c = ch0; c < ch1; c += 8) {
      const int kg = c >> 3, chunk = kg / g.kgs, k = kg - chunk * g.kgs;
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
                                                 irsrc, inside && c + q < ch1 ? at + q * hw4 : kOutside, 0, 0));
          const u32x4* d = block + (size_t)((chunk * g.ks * g.ks + r * g.ks + s) * halves + (k >> 1)) * 192 + (k & 1) * 32 + 4 * (again >> 5);
#pragma unroll
          for (int j = 0; j < 16 / KW; ++j) {
            const int i = team * (16 / KW) + j, row = 8 * (i / 4) + i % 4;
            const u32x4 h = d[row], m = d[row + 64], l = d[row + 128];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
              auto part = [&](u32x4 x) { return __builtin_bit_cast(float, q & 1 ? x[q / 2] & 0xffff0000u : x[q / 2] << 16); };
              const float w = part(h) + part(m) + part(l);
              if (w != 0.f) sum[j] = fmaf(v[q], w * (1 / kScale), sum[j]);
            }
          }
        }
    }
#pragma unroll
    for (int j = 0; j < 16 / KW; ++j) store(team * (16 / KW) + j, b, sum[j]);
  }
}

// packed streams -> the weights' parts in the order the matrix kernel's lanes load them; one wave per stream
__global__ __launch_bounds__(256) void parts_kernel(const int32_t* __restrict__ grp_off, const int32_t* __restrict__ grp_nnz,
                                                    const int32_t* __restrict__ oc_order, const int32_t* __restrict__ position,
                                                    const float* __restrict__ values, unsigned short* __restrict__ dst, int K,
                                                    int ks, int tile_ic, int stages, int G, int nstream, int kgs, int steps) {
  const int sid = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (sid >= nstream) return;
  const int grp = sid / stages, st = sid - grp * stages;
  const int beg = grp_off[sid], n = grp_nnz[sid];
  for (int i = lane; i < n; i += 64) {
    const unsigned pos = (unsigned)position[beg + i];
    const float v = values[beg + i];
    const int s = pos & 7, r = (pos >> 3) & 7, ic = st * tile_ic + (int)((pos >> 6) & 0x3ffff);
    const int oc = oc_order[grp * G + (int)(pos >> 24)];
    if (oc < 0 || oc >= K) continue;
    const int kg = ic >> 3, chunk = kg / kgs, k = kg - chunk * kgs;
    const int step = (chunk * ks * ks + r * ks + s) * (kgs >> 1) + (k >> 1);
    unsigned short* d = dst + (((size_t)(oc >> 5) * steps + step) * 192 + (k & 1) * 32 + (oc & 31)) * 8 + (ic & 7);
    float x[8] = {v, 0, 0, 0, 0, 0, 0, 0};
    u32x4 h, m, l;
    cut(x, h, m, l);
    d[0] = (unsigned short)h[0];
    d[512] = (unsigned short)m[0];
    d[1024] = (unsigned short)l[0];
  }
}

// input buffers, or what the teams' sums need
int lds_main(const MatGeom& g) {
  const MatShape& c = kMatShapes[g.cfg];
  return std::max(c.kw * 96 * g.kgs * g.lpad, c.kw > 1 ? c.kw * c.wm * c.wn * 4096 * c.nb : 0);
}
int lds_bytes(const MatGeom& g) { return lds_main(g) + (g.half ? 128 * kMatShapes[g.cfg].wm + kAsideBytes : 0); }

template <int WM, int NB, int KW, int TM>
int launch_one(const MatGeom& g, const float* d_in, float* d_out, const void* weights, hipStream_t stream) {
  auto kern = matrix_kernel<WM, NB, KW, TM>;
  static std::atomic<bool> lds_set{false};  // per instantiation; setting the attribute twice is harmless
  if (!lds_set.load(std::memory_order_acquire)) {
    TETRIS_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kMatLds));
    lds_set.store(true, std::memory_order_release);
  }
  const int grid = 8 * ceil_div(g.ptiles * g.mtiles * g.csplit, 8);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(256 * KW), lds_bytes(g), stream, d_in, d_out,
                     static_cast<const u32x4*>(weights), g);
  TETRIS_HIP(hipGetLastError());
  return TETRIS_OK;
}

MatDiv divider(int d) {
  MatDiv r{};
  int l = 0;
  while ((1 << l) < d) ++l;
  r.shift = 30 + l;
  r.m = (unsigned)(((1ull << r.shift) + (unsigned)d - 1) / (unsigned)d);
  return r;
}

// staged pixels the largest tile of `P` pixels needs
int staged_pixels(const MatGeom& g, int P) {
  const int psh = g.pool ? 2 : 0, dbl = g.pool ? 1 : 0;
  auto at = [&](int u, int d) {
    const int q = u / g.upq, r = u - q * g.upq, y = r / g.uw, x = r - y * g.uw;
    return ((long long)q * g.ihs + (long long)((y << dbl) + d) * g.stride) * g.wp + (long long)((x << dbl) + d) * g.stride;
  };
  // (the tiles' starts repeat, relative to their strip, after upq / gcd tiles at the latest)
  const int per = P >> psh, tiles = std::min(ceil_div(g.npix, P), g.upq / std::gcd(per, g.upq));
  long long most = 0;
  for (int t = 0; t < tiles; ++t)
    most = std::max(most, at(t * per + per - 1, dbl) - at(t * per, 0) + (long long)(g.ks - 1) * (g.wp + 1) + 1);
  return (int)std::min<long long>(most, 1 << 28);
}

}  // namespace

// Cuts a layer into workgroups of configuration `cfg` with `csplit` slices of the channels; false: it cannot be run so.
bool make_mat_geom(int N, int C, int H, int W, int K, int ks, int stride, int pad, int cfg, int csplit, bool pool, MatGeom* out,
                   StagedPixels* staged) {
  MatGeom g{};
  if (N <= 0 || C <= 0 || H <= 0 || W <= 0 || K <= 0 || cfg < 0 || cfg >= kMatConfigs || csplit < 1 || csplit > kMaxSplit) return false;
  g.N = N; g.C = C; g.H = H; g.W = W; g.K = K; g.ks = ks; g.pad = pad;
  g.OH = out_extent(H, pad, ks, stride);
  g.OW = out_extent(W, pad, ks, stride);
  if (g.OH < 1 || g.OW < 1 || H + 2 * pad < ks || W + 2 * pad < ks || (pool && (g.OH < 2 || g.OW < 2))) return false;
  g.sub = ks == 1 ? stride : 1;  // a pointwise layer reads every stride-th row and column only
  g.stride = ks == 1 ? 1 : stride;
  // 32-bit byte offsets below kOutside
  if (4ll * N * C * H * W >= (1ll << 30) || 4ll * N * K * g.OH * g.OW >= (1ll << 30)) return false;
  g.in_bytes = 4 * N * C * H * W;
  g.pool = pool;
  g.out_floats = pool ? N * K * (g.OH / 2) * (g.OW / 2) : N * K * g.OH * g.OW;
  // Images wider than 64 are cut into strips, which are images to everything below: a tile's pixels are consecutive in a
  // strip, row by row, and the rows above and below that it stages as well are a strip wide.
  g.strips = ceil_div(g.OW, 64);
  g.ws = ceil_div(g.OW, g.strips);
  if (g.strips > 1 || pool) g.ws += g.ws & 1;
  if (pool && g.strips == 1) g.ws = g.OW & ~1;
  g.wp = (g.ws - 1) * g.stride + ks;
  g.ihs = (g.OH - 1) * g.stride + ks;
  g.uw = pool ? g.ws / 2 : g.ws;
  g.uh = pool ? g.OH / 2 : g.OH;
  g.upq = g.uw * g.uh;
  if ((long long)N * g.strips * g.upq * (pool ? 4 : 1) >= (1ll << 30)) return false;
  g.npix = N * g.strips * g.upq * (pool ? 4 : 1);
  g.half = kMatShapes[cfg].half;
  g.kgs = ks == 1 ? 4 : 2;
  if (g.half) {
    if (C > kMostChannels) return false;
    // (A step's words have room for 8 groups, and for 2 where ks > 4.)  Long chunks: fewer barriers, and fewer steps that are not
    // full; short ones: more workgroups on a CU, and tiles whose halo would not fit else.
    g.kgs = C <= 16 || ks > 4 ? 2 : C <= 32 || ks > 1 ? 4 : 8;
    if (kMatShapes[cfg].brief) {
      if (g.kgs == 2) return false;
      g.kgs /= 2;
    }
  }
  g.chunks = ceil_div(C, 8 * g.kgs);
  if (csplit > g.chunks) return false;
  g.csplit = csplit;
  g.steps = g.chunks * ks * ks * (g.kgs / 2);
  g.mblocks = ceil_div(K, 32);
  const MatShape c = kMatShapes[cfg];
  g.cfg = cfg;
  g.smax = ceil_div(2 * g.kgs * ks * ks, 4);
  if (g.half && (g.chunks / csplit < c.kw || ((long long)g.mblocks * g.chunks * g.smax + 3) * kStepBytes >= (1ll << 31))) return false;
  const int P = 32 * c.nb * c.wn;
  g.ptiles = ceil_div(g.npix, P);
  g.mtiles = ceil_div(g.mblocks, c.wm);
  StagedPixels one{};
  int& most = (staged ? *staged : one)[P / 32];
  if (!most) most = staged_pixels(g, P);
  g.lpad = ceil_div(most, 64) * 64;
  if (g.kgs * g.lpad / 64 > c.wm * c.wn * (g.half && c.nb == 4 ? 2 : kMatTasks) || lds_bytes(g) > kMatLds) return false;
  g.lds_rows = lds_main(g);
  if ((long long)g.ptiles * g.mtiles * csplit >= (1ll << 28)) return false;
  // multiply-high divisions: dividend * divisor below 2^32
  const long long lim = 1ll << 32;
  if ((long long)(g.uw + P) * g.uw >= lim || (long long)(g.uh + P) * g.uh >= lim ||
      (long long)(g.wp + g.lpad) * g.wp >= lim || (long long)(g.ihs + g.lpad) * g.ihs >= lim ||
      (long long)(N * g.strips + P + g.lpad) * g.strips >= lim)
    return false;
  g.m_uw = magic_reciprocal(g.uw); g.m_uh = magic_reciprocal(g.uh); g.m_wp = magic_reciprocal(g.wp);
  g.m_ihs = magic_reciprocal(g.ihs); g.m_strips = magic_reciprocal(g.strips);
  g.d_tiles = divider(g.ptiles * g.mtiles); g.d_mtiles = divider(g.mtiles); g.d_upq = divider(g.upq);
  g.d_uw = divider(g.uw); g.d_blocks = divider(g.lpad / 64);
  *out = g;
  return true;
}

// Microseconds of a launch.  The constants were fitted to the times of a kernel with six products a step, whose cycles
// were then scaled by 8/6.  Against 13 462 timed launches of 424 layers -- those of the benchmark's suites at batch 1, 4
// and 16 and 160 random ones, every configuration and slice count: profiles/kernel_times.txt, measured and checked by
// tetris_amd/kernel_times.py -- they are 11 % off (standard deviation).  A fit to these times, with a term for the weights'
// bytes, is 11 % off as well and not faster in any network (VGG19 at batch 1: 408 us, 400 with these).
double plain_time(const MatGeom& g) {
  const MatShape& c = kMatShapes[g.cfg];
  const int by_regs = c.nb == 4 ? 2 / c.kw : c.nb == 2 ? std::max(1, 3 / c.kw) : c.kw == 1 ? 5 : c.kw == 2 ? 2 : 1;
  const int fit = std::max(1, std::min(by_regs, kMatLds / lds_bytes(g)));  // workgroups per CU
  const int wgs = g.ptiles * g.mtiles * g.csplit, rounds = ceil_div(ceil_div(g.chunks, g.csplit), c.kw);
  const int steps = g.ks * g.ks * g.kgs / 2, staging = ceil_div(g.kgs * g.lpad, 256);
  // cycles of n workgroups on a CU: start and end; a round's staging and barrier; a step, which waits for its weights or,
  // with enough waves, for the matrix core (8 * nb products of 32 cycles per team and SIMD)
  auto cycles = [&](int n) {
    if (n == 0) return 0.0;
    const double step = std::max(g.ks == 1 ? 193.0 : 539.0, 1.205 * 256 * c.nb * c.kw * n);
    return 3958.0 + 349.0 * c.nb * n * c.kw + rounds * ((g.ks == 1 ? 1031.0 : 2033.0) + 321.0 * staging * c.kw * n + steps * step);
  };
  const int full = wgs / (256 * fit), rest = wgs % (256 * fit);
  const double compute = (full * cycles(fit) + cycles(ceil_div(rest, 256))) / 2.2e3;
  const double out = 4.0 * g.N * g.K * g.OH * g.OW, in = 4.0 * g.N * g.C * (g.ks == 1 ? g.OH : g.H) * g.W;
  const double memory = (in * (1 + 0.19 * std::sqrt(g.mtiles - 1.0)) + out * g.csplit) / 4.17e6;
  return 2.2 + std::max(compute, memory) + (g.csplit > 1 ? 2.5 + out * (g.csplit + 1) / 4.07e6 : 0);
}

// The same for half_kernel, fitted to launches of the same layers before inputs out of range were listed: 9 % off on 13 749 since.
double half_time(const MatGeom& g, long long nnz) {
  const MatShape& c = kMatShapes[g.cfg];
  const int team = c.wm * c.wn, waves = team * c.kw;
  const int by_regs = std::max(1, (c.nb >= 2 ? 8 : 12) / waves);
  const int fit = std::max(1, std::min(by_regs, kMatLds / lds_bytes(g)));  // workgroups per CU
  const int wgs = g.ptiles * g.mtiles * g.csplit, rounds = ceil_div(ceil_div(g.chunks, g.csplit), c.kw);
  // steps of a chunk: its blocks, those of them again that hold more than two weights in a group of four, four to a step
  const double density = std::min(1.0, (double)nnz / ((double)g.K * g.C * g.ks * g.ks)), more = density * density * density * (4 - 3 * density);
  const double blocks = (double)ceil_div(g.C, 8) * g.ks * g.ks / g.chunks, staging = (double)g.kgs * g.lpad / 64 / team;
  const double steps = blocks * (2 - std::pow(1 - more, 64)) / 4 + 0.375;
  // cycles of n workgroups on a CU: start and end; a round's staging and barrier; a step, as long as one wave takes or, with
  // enough waves, the matrix core (6 * nb products of 32 cycles per wave)
  auto cycles = [&](int n) {
    if (n == 0) return 0.0;
    const double per_simd = n * waves / 4.0, products = 192.0 * c.nb;
    const double step = std::max(165.0 + 2.032 * products, (87.0 + 1.231 * products) * per_simd);
    return 4973.0 + 1257.0 * c.nb * per_simd + rounds * ((g.ks == 1 ? 221.0 : 722.0) + 681.0 * staging * per_simd + steps * step);
  };
  const int full = wgs / (256 * fit), rest = wgs % (256 * fit);
  const double out = 4.0 * g.N * g.K * g.OH * g.OW;
  return 1.67 + (full * cycles(fit) + cycles(ceil_div(rest, 256))) / 2.3e3 + (g.csplit > 1 ? 2.48 + out * (g.csplit + 1) / 4.3e6 : 0);
}

double matrix_time(const MatGeom& g, long long nnz) { return g.half ? half_time(g, nnz) : plain_time(g); }

// The same for the kernels that walk the non-zeros: 15 % off.
double walk_time(const Geom& g, long long nnz) {
  const int family = g.ver - 2;  // one LDS tile, three LDS buffers, flat
  constexpr double start[] = {12362, 12723, 9370}, stage[] = {2346, 5171, 1186}, busy[] = {1.872, 0.955, 1.442}, alone[] = {60.8, 55.6, 60};
  const double entry = g.nq == 1 ? 26.2 : g.nq == 2 ? 43.5 : 85.0;  // cycles of an entry on a full SIMD
  const double entries = ((double)nnz / g.K * g.g + 1.05 * g.stages) / g.csplit;  // of a wave, with its padding
  const int fit = g.waves == 16 || (g.waves == 8 && g.buf_bytes != kHalfBufBytes && g.buf_bytes != kFlatHalfBufBytes) ? 1 : 2;
  auto cycles = [&](int n) {
    if (n == 0) return 0.0;
    return start[family] + stage[family] * g.stages / g.csplit +
           std::max(entries * n * g.waves / 4 * entry * busy[family], entries * alone[family] * std::sqrt((double)g.nq));
  };
  const int wgs = g.ugroups * g.kblocks * g.csplit, full = wgs / (256 * fit), rest = wgs % (256 * fit);
  const double compute = (full * cycles(fit) + cycles(ceil_div(rest, 256))) / 2.3e3;
  const double out = 4.0 * g.N * g.K * g.OH * g.OW, in = 4.0 * g.N * g.C * g.H * g.W;
  return std::max(compute, (in + out) / 6.9e6) + (g.csplit > 1 ? 1.5 + out * (g.csplit + 1) / 4.1e6 : 0);
}

// Whether a matrix kernel is worth running in place of the walking kernel of geometry `walk`, and how: the configuration and slice
// count of least predicted time, if that is 7 % below the walking kernel's; half_kernel's, if that is 16 % below the walking
// kernel's -- predictions for large walks are 8 % too long -- and 5 % below matrix_kernel's.  Of the 424 timed layers 125
// then go to matrix_kernel and 96 to half_kernel; over all of them that is 1.192 times the walk's speed, 3.0 % short of the
// best choice.  10 layers lose more than 3 % to the walk, all on matrix_kernel and pointwise or of one image, two of them half
// as much again (1 x 512 -> 1024 28x28 15.6 us, 10.6; 1 x 1024 -> 255 13x13 15.4, 10.5; with 10 % instead of 7 % two layers lose, 9 % at
// most, and 1.191 times), and six to what matrix_kernel and the walk alone would give them.  (Without half_kernel 1.152 times.  With
// 12 % to the walk 13 layers lose so, with 10 % and no advantage asked over matrix_kernel 27.)  Where the walking kernel can pool its
// outputs, so must the matrix kernel.
bool choose_mat_geom(int N, int C, int H, int W, int K, int ks, int stride, int pad, const Geom& walk, long long nnz,
                     MatGeom* g, MatGeom* pool) {
  if (C < 16) return false;  // most of a chunk of 16 channels would be padding
  const bool pools = walk.OH >= 2 && walk.OW >= 2 && (walk.csplit > 1 || geom_pools_in_kernel(walk));
  struct Found { double t; int cfg, slices; };
  std::vector<Found> found;
  StagedPixels staged{};
  const double walking = walk_time(walk, nnz);
  for (int cfg = 0; cfg < kMatConfigs; ++cfg) {
    MatGeom m;
    if (!make_mat_geom(N, C, H, W, K, ks, stride, pad, cfg, 1, false, &m, &staged)) continue;
    for (const int slices : {1, 2, 3, 4, 6, 8}) {
      if (m.chunks / slices < (m.half ? kMatShapes[cfg].kw : 1) || (slices > 1 && 4ll * m.out_floats * slices > kMatCopies)) break;
      m.csplit = slices;
      const double t = matrix_time(m, nnz);
      if (t < (m.half ? 0.84 : 0.93) * walking) found.push_back({m.half ? 1.05 * t : t, cfg, slices});
    }
  }
  std::stable_sort(found.begin(), found.end(), [](const Found& a, const Found& b) { return a.t < b.t; });
  for (const Found& f : found) {
    *pool = MatGeom{};
    if (f.slices == 1 && walk.OH >= 2 && walk.OW >= 2 && !make_mat_geom(N, C, H, W, K, ks, stride, pad, f.cfg, 1, true, pool)) {
      *pool = MatGeom{};
      if (pools) continue;
    }
    return make_mat_geom(N, C, H, W, K, ks, stride, pad, f.cfg, f.slices, false, g, &staged);
  }
  return false;
}

int mat_lds_bytes(const MatGeom& g) { return lds_bytes(g); }

size_t mat_weight_bytes(const MatGeom& g) { return g.half ? half_weight_bytes(g) : (size_t)g.mblocks * g.steps * 192 * 16; }

int mat_weights(const tetris_g950* p, const MatGeom& g, hipStream_t stream, void* dst, MatWeights* out) {
  if (g.half) return half_weights(p, g, stream, dst, out);
  TETRIS_HIP(hipMemsetAsync(dst, 0, mat_weight_bytes(g), stream));
  const int nstream = p->groups * p->stages;
  hipLaunchKernelGGL(parts_kernel, dim3(ceil_div(nstream, 4)), dim3(256), 0, stream, p->d_grp_off, p->d_grp_nnz, p->d_oc_order,
                     p->d_position, p->d_values, static_cast<unsigned short*>(dst), p->K, p->ks, p->tile_ic, p->stages, p->g,
                     nstream, g.kgs, g.steps);
  TETRIS_HIP(hipGetLastError());
  TETRIS_HIP(hipStreamSynchronize(stream));  // launches on other streams may follow at once
  *out = MatWeights{};
  out->base = dst;
  return TETRIS_OK;
}

int launch_matrix(const MatGeom& g, const float* d_in, float* d_out, const MatWeights& w, int relu, hipStream_t stream) {
  if (g.half) return launch_half(g, d_in, d_out, w, relu, stream);
  const void* weights = w.base;
  MatGeom k = g;
  k.relu = relu;
  k.quads = stores_quads(g, d_out);
  const bool two = g.kgs * g.lpad / 64 <= 8;
#define TETRIS_MAT(WM, NB, KW) \
  if (c.wm == WM && c.nb == NB && c.kw == KW) \
    return two ? launch_one<WM, NB, KW, 2>(k, d_in, d_out, weights, stream) : launch_one<WM, NB, KW, kMatTasks>(k, d_in, d_out, weights, stream);
  const MatShape& c = kMatShapes[g.cfg];
  TETRIS_MAT(4, 4, 1) TETRIS_MAT(4, 4, 2) TETRIS_MAT(4, 2, 1) TETRIS_MAT(4, 2, 2) TETRIS_MAT(4, 2, 4) TETRIS_MAT(2, 2, 1)
  TETRIS_MAT(2, 2, 2) TETRIS_MAT(2, 2, 4) TETRIS_MAT(2, 1, 1) TETRIS_MAT(2, 1, 2) TETRIS_MAT(2, 1, 4)
#undef TETRIS_MAT
  return fail(TETRIS_EINVAL, "no matrix kernel of configuration %d", g.cfg);
}

}  // namespace tetris
