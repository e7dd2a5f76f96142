// Sparse convolution on the matrix cores with three products of fp16 parts a weight, for the layers that the walk would run else.
//
// An input is two fp16 parts, x = a + 2^-11 b: rounded to eleven bits, and what that leaves, rounded likewise.  A weight is the sum of
// `near`, to eleven bits, and `off`.  The products off * a, near * a and (2^-11 near) * b are summed in fp32 (off * b, 2^-22 of the
// product, is left out); half_kernel has six, of three parts, and is more exact: 6.8e-8 to 9.4e-8 of the outputs' 2-norm, where this
// kernel is off by 1.1e-7 (115 terms) to 1.7e-7 (790) and the walk by 1.4e-7 to 3.6e-7 -- what the matrix core drops when it adds counts
// more than the parts.  So it takes layers from the walk alone, and only where the walk's sums are long (choose_mat_geom).
//
// What bounds it is issue.  A product is 33 cycles of a SIMD, but a wave that reads its inputs, decodes their places and asks for weights
// between products keeps the matrix core half busy; two waves fill it up to 5 VALU instructions or 2 LDS reads a product and wave.  So all
// eight waves of a workgroup, which has a CU to itself, multiply, four blocks of 32 pixels each -- a step's weights, 2.3 KiB from L2, meet
// 12 products, and a step takes 1100 to 1350 cycles of two waves, whose products alone are 792 -- and in between they stage what is
// multiplied next: the first chunk of the next tile too, so that of the 18 000 cycles that a workgroup takes to its first product
// (tiles, the inputs' scale, two trips to memory, a barrier) a run of tiles pays once.  The halves of the workgroup, of which a SIMD has one
// wave each, stage at different times, and no barrier ends a chunk (Stage::arrive): a wave whose channels have fewer steps goes ahead of the others
// by up to a third of one, 141 against 134 us on 16 x 512 -> 512 28x28, 78 against 77 on 16 x 256 -> 512 26x26.  Sums are cleared every eight steps into a second set that is rounded less often: 1.92e-7 becomes
// 1.49e-7 on 16 x 512 -> 512 28x28 (with the two kinds of small products summed apart instead 2.3e-7; clearing every two steps 1.89e-7).
//
// Microseconds, the walk and this: 16 x 256 -> 256 56x56, 10 % of the weights, 159 and 132 to 140 (large layers run at 1.5 to 1.8 GHz here,
// held back by power); 15 % 222 and 163; 16 x 512 -> 512 28x28 175 and 128 to 136; 16 x 256 -> 512 26x26, 15 %, 124 and 71; 9 x 157 -> 152 134x134
// 5x5, 20 %, 1060 and 633.  Half of the waves staging for the others, which then multiply twelve blocks a step, took 5 to 20 % longer, and so
// did one loop for all counts of blocks in a tile.
#include "matrix_half.h"

namespace tetris {
namespace {

constexpr int kWaves = 8;  // of a workgroup
constexpr int kTile = 4;   // most blocks of 32 pixels of a tile, of a wave

// Two fp16 parts of eight floats, scaled: the number rounded to eleven bits, and 2^11 times what that leaves, rounded likewise.
__device__ __forceinline__ void cut2(const float (&x)[8], float scale, u32x4& hi, u32x4& lo, f16x2& zeros) {
  const float scale_rest = scale * kRest;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = x[2 * i], b = x[2 * i + 1];
    const f16x2 h = __builtin_convertvector((f32x2{a * scale, b * scale}), f16x2);
    const float r0 = fmaf((float)h.x, -kRest, a * scale_rest), r1 = fmaf((float)h.y, -kRest, b * scale_rest);
    zeros = __builtin_elementwise_fma(h, f16x2{0, 0}, zeros);
    hi[i] = __builtin_bit_cast(unsigned, h);
    lo[i] = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{r0, r1}), f16x2));
  }
}

// What a workgroup does: of 32*WM output channels and a slice of the input channels a run of pixels, tile after tile.
struct Work {
  int slice, mt, c_beg, rounds;  // rounds: chunks of the slice, from c_beg on
  int first, blocks, tiles;      // blocks of 32*WN pixels, cut into tiles of four and three, seldom two
  int shared;                    // of the run's blocks the last is the next run's, too (1), or the first that of the run before (2): see own_of
};
struct Tile {
  int block, count;                 // first block of pixels and how many
  int q0, oy0, ox0, row0, col0;     // first pixel: strip image, row and column in it; row and column of the first staged one
  int staged;                       // quads of staged pixels
};

__device__ __forceinline__ Work work_of(Arguments arguments) {
  const auto& g = arguments->g;
  // workgroup ids go round-robin to the XCDs: each XCD gets a contiguous range of logical ids.  Channel blocks of one run of
  // pixels are neighbours (they read the same input), slices outermost (they share nothing).
  const int id = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  Work w;
  const int all = g.runs * g.mtiles;
  w.slice = quotient(id, g.d_tiles);
  const int run = quotient(id - w.slice * all, g.d_mtiles);
  w.mt = id - w.slice * all - run * g.mtiles;
  w.c_beg = w.slice * g.chunks / g.csplit;
  w.rounds = (w.slice + 1) * g.chunks / g.csplit - w.c_beg;
  const int rest = g.run_rest << g.run_halves;
  w.first = run * g.run_blocks + (min(run, rest) >> g.run_halves);
  w.blocks = g.run_blocks + (run < rest);
  w.shared = g.run_halves && run < rest ? 1 + (run & 1) : 0;
  w.tiles = (w.blocks + kTile - 1) / kTile;
  return w;
}

template <int WN>
__device__ __forceinline__ Tile tile_of(Arguments arguments, const Work& w, int k) {
  const auto& g = arguments->g;
  Tile t;
  // (Tiles of four, the last ones of three; a run of five of three and two, and a single block as two of which one is left out.)
  const int short_by = kTile * w.tiles - w.blocks, threes = k - (w.tiles - short_by);
  if (w.tiles >= short_by) {
    t.block = w.first + kTile * k - max(threes, 0);
    t.count = threes < 0 ? kTile : kTile - 1;
  } else {
    t.block = w.first + (kTile - 1) * k;
    t.count = max(min(w.blocks - (kTile - 1) * k, kTile - 1), 2);
  }
  const int psh = g.pool ? 2 : 0, dbl = g.pool ? 1 : 0;
  auto at = [&](int u, int& q, int& y, int& x) {
    q = quotient(u, g.d_upq);
    const int r = u - q * g.upq;
    y = quotient(r, g.d_uw);
    x = r - y * g.uw;
  };
  at((t.block * 32 * WN) >> psh, t.q0, t.oy0, t.ox0);
  t.row0 = (t.oy0 << dbl) * g.stride;
  t.col0 = (t.ox0 << dbl) * g.stride & ~3;
  int q, y, x;
  at(min((t.block + t.count) * 32 * WN >> psh, g.npix >> psh) - 1, q, y, x);
  const int last = ((q - t.q0) * g.ihs + ((y << dbl) + dbl) * g.stride - t.row0) * g.wp + ((x << dbl) + dbl) * g.stride - t.col0;
  t.staged = (last + (g.ks - 1) * (g.wp + 1) + 4) >> 2;
  return t;
}

// Which blocks of a tile a wave multiplies and which of them it stores.  Where runs are a block longer than others, a launch takes as long as
// if all were.  So two neighbours share a block instead, each for half of the output channels: the first for those of its first four waves, the
// second for those of the others.  (A SIMD has one wave of each half.)  Microseconds before and with it: 126 and 120 on 16 x 512 -> 512 28x28,
// 10 % of the weights (128 runs of 3 blocks for each half of the channels, 8 of which had 4), 111 and 107 on 16 x 256 -> 256 48x48 (4.5 blocks), 134 and 132 on
// 56x56 (6.125): power holds the others back while all CUs are busy.  Where more than half of the runs have one more there is nothing to share.
struct Own { int first, count, stores; };  // stores: a bit each
__device__ __forceinline__ Own own_of(const Work& w, const Tile& t, int k, int wave) {
  const bool half = wave >= kWaves / 2;
  const int lead = w.shared == 2 && !half && k == 0, trail = w.shared == 1 && half && k == w.tiles - 1;
  const int stored = t.count - lead - trail;
  if (stored < 2) return {0, t.count, ((1 << stored) - 1) << lead};
  return {lead, stored, (1 << stored) - 1};
}

// The geometry's numbers that places are worked out with, read at once: each first touch of a line is a trip to L2.
struct Places { unsigned m_uw, m_uh, m_wp, m_ihs, m_strips; int uw, uh, wp, ihs, strips, ws, stride, sub, pad, pool, npix, H, W, C, N, ks, kgs, lpad; };
__device__ __forceinline__ Places places_of(Arguments arguments) {
  const auto& g = arguments->g;
  return {g.m_uw, g.m_uh, g.m_wp, g.m_ihs, g.m_strips, g.uw, g.uh, g.wp, g.ihs, g.strips, g.ws, g.stride, g.sub, g.pad, g.pool, g.npix, g.H, g.W, g.C, g.N, g.ks, g.kgs, g.lpad};
}

constexpr int kNone = 1 << 30;  // behind every input, which are smaller
// Where the staged pixels 4 i to 4 i + 3 of a tile lie in its first channel, in bytes, and which of them lie in the image.  (Below zero: the
// tensor's first pixels, with columns outside of the image before them.  None: far behind every input.)
__device__ __forceinline__ int source_of(const Places& at, const Tile& t, int i, unsigned& inside) {
  const unsigned x = t.col0 + 4 * i;
  const unsigned dr = over(x, at.m_wp), col = x - dr * at.wp;
  const unsigned row = t.row0 + dr;
  const unsigned dq = over(row, at.m_ihs), y = row - dq * at.ihs;
  const unsigned q = t.q0 + dq, n = over(q, at.m_strips), strip = q - n * at.strips;
  const int iy = (int)y - at.pad, ix = (int)(strip * at.ws * at.stride + col) - at.pad;
  inside = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) inside |= ix + e >= 0 && ix + e < at.W ? 1u << e : 0;
  if (n >= (unsigned)at.N || iy < 0 || iy >= at.H) inside = 0;
  return inside ? 4 * (int)(n * (unsigned)(at.C * at.H * at.W) + (unsigned)(iy * at.W + ix)) : kNone;
}

// where a lane's pixel of block `b` of a tile lies: in the output's images, in LDS and in the output
struct Pixel { bool in_range; int t; unsigned n, dq, uy, oy, ox, w; };  // ox: in its strip, w: in its image
template <int WN>
__device__ __forceinline__ Pixel pixel_of(const Places& at, const Work& w, const Tile& tile, int block, int lane) {
  const int psh = at.pool ? 2 : 0, dbl = at.pool ? 1 : 0;
  Pixel p;
  // (16 pixels side by side are read at a time: by four lanes each of 0-3, 12-15, 20-27, and of 4-11, 16-19, 28-31)
  const int t = block * 32 + (0x73261540 >> (lane & 28) & 7) * 4 + (lane & 3), beg = tile.block * 32 * WN;
  const int end = min(at.npix, (w.first + w.blocks) * 32 * WN);
  p.in_range = beg + t < end;
  p.t = p.in_range ? t : end - 1 - beg;
  const unsigned x = tile.ox0 + (p.t >> psh);
  const unsigned dy = over(x, at.m_uw), ux = x - dy * at.uw, y = tile.oy0 + dy;
  p.dq = over(y, at.m_uh);
  p.uy = y - p.dq * at.uh;
  p.oy = (p.uy << dbl) + (at.pool ? (p.t >> 1) & 1 : 0);
  p.ox = (ux << dbl) + (at.pool ? p.t & 1 : 0);
  const unsigned q = tile.q0 + p.dq;
  p.n = over(q, at.m_strips);
  p.w = (q - p.n * at.strips) * at.ws + p.ox;
  return p;
}
__device__ __forceinline__ int lds_of(const Places& at, const Tile& tile, const Pixel& p) {
  return ((int)(p.dq * at.ihs + p.oy * at.stride) - tile.row0) * at.wp + (int)p.ox * at.stride - tile.col0;
}
__device__ __forceinline__ int out_of(Arguments arguments, const Pixel& p, int lane) {
  const auto& g = arguments->g;
  if (g.pool)
    return p.in_range && (p.t & 3) == 0 && (p.w >> 1) < (unsigned)(g.OW >> 1)
               ? 4 * (int)((p.n * g.K + 4 * (lane >> 5)) * ((g.OH >> 1) * (g.OW >> 1)) + p.uy * (g.OW >> 1) + (p.w >> 1)) : kOutside;
  return p.in_range && p.w < (unsigned)g.OW ? 4 * (int)((p.n * g.K + 4 * (lane >> 5)) * (g.OH * g.OW) + p.oy * g.OW + p.w) : kOutside;
}

// Sums i to i + 3 of a lane are channels 8*(i/4) + 4*(lane/32) + 0..3 of its wave's 32, of one pixel.
struct Stores {
  __amdgpu_buffer_rsrc_t rsrc;
  int oc0, ohw, K, pool, relu, quads;
};
__device__ __forceinline__ Stores stores_of(Arguments arguments, const Work& w, int oc0) {
  const auto& g = arguments->g;
  return {__builtin_amdgcn_make_buffer_rsrc(arguments->out + (size_t)w.slice * g.out_floats, 0, 4 * g.out_floats, 0x00020000), oc0,
          g.pool ? (g.OH >> 1) * (g.OW >> 1) : g.OH * g.OW, g.K, g.pool, g.relu, g.quads};
}
__device__ __forceinline__ void store(const Stores& s, int lane, int i, int off, float (&v)[4]) {
  if (s.quads) {
    // four pixels of a channel to a lane instead of four channels of a pixel: a store of 16 bytes instead of four
    transpose_quad(v, lane);
    u32x4 d;
#pragma unroll
    for (int k = 0; k < 4; ++k) d[k] = bits_of(s.relu ? fmaxf(v[k], 0.f) : v[k]);
    __builtin_amdgcn_raw_buffer_store_b128(d, s.rsrc, s.oc0 + 2 * i + 4 * (lane >> 5) + (lane & 3) < s.K && off != kOutside ? off + 4 * (lane & 3) * (s.ohw - 1) : kOutside,
                                           (s.oc0 + 2 * i) * s.ohw * 4, 0);
    return;
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int oc = s.oc0 + 2 * i + k;
    float d = s.pool ? quad_max(v[k]) : v[k];
    if (s.relu) d = fmaxf(d, 0.f);
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, d), s.rsrc, oc + 4 * (lane >> 5) < s.K ? off : kOutside, oc * s.ohw * 4, 0);
  }
}

constexpr int kBytes = kStepBytes2;  // of a step
struct Step { u32x4 p[2]; unsigned word; };
struct Weights {
  __amdgpu_buffer_rsrc_t rsrc;
  int lane;
};
__device__ __forceinline__ void fetch(const Weights& w, int step, Step& s) {
#pragma unroll
  for (int p = 0; p < 2; ++p) s.p[p] = __builtin_amdgcn_raw_buffer_load_b128(w.rsrc, w.lane * 16, step * kBytes + p * 1024, 0);
  s.word = __builtin_amdgcn_raw_buffer_load_b32(w.rsrc, w.lane * 4, step * kBytes + 2048, 0);
}

// What lies in LDS behind the staged inputs, for three tiles at a time: while one is multiplied, the first chunk of the next one is staged, and
// values that tell the scale of the one after it are read.
struct Shared {
  int* shift;        // [4] inputs of a tile are multiplied by two to this
  unsigned* most;    // [3][kWaves] the largest of a few of them, per wave
  unsigned* asides;  // [3][16] per wave: how many inputs are set aside; 8: whether they are too many after the first chunk
  int* counts;       // [2] chunks that waves have staged, all waves' added up, from a workgroup's second on; chunks that they have multiplied
  int2* aside;       // [3][kWaves][kMostAside] ... which: channel and staged pixel; the input
  float* sums;       // [kWaves][1024] of a block of pixels
};
__device__ __forceinline__ Shared shared_of(Arguments arguments, u32x4* lds) {
  Shared s;
  s.shift = reinterpret_cast<int*>(reinterpret_cast<char*>(lds) + arguments->g.lds_rows);
  s.most = reinterpret_cast<unsigned*>(s.shift + 4);
  s.asides = s.most + 3 * kWaves;
  s.counts = reinterpret_cast<int*>(s.asides + 48);
  s.aside = reinterpret_cast<int2*>(s.counts + 2);
  s.sums = reinterpret_cast<float*>(s.aside + 3 * kWaves * kMostAside);
  return s;
}
static_assert(kRelayBytes == 4 * 4 + 3 * kWaves * 4 + 48 * 4 + 2 * 4 + 3 * kWaves * kMostAside * 8);
constexpr int kPart = kRelayPart / 16;  // A part of all staged inputs lies a fixed distance from the other, which reads have room for in their offsets.

// whether a tile that is all staged has more inputs set aside than are multiplied one by one
__device__ __forceinline__ bool too_many(const Shared& s, int slot, int lane) {
  const unsigned listed = s.asides[16 * slot + lane / kMostAside];
  return __builtin_popcountll(__builtin_amdgcn_ballot_w64(lane % kMostAside < listed)) > (int)kMostAside ||
         __builtin_amdgcn_ballot_w64(listed > kMostAside);
}
__device__ __forceinline__ bool too_many_soon(const Shared& s, int slot, int lane) {
  return __builtin_amdgcn_ballot_w64(s.asides[16 * slot + 8 + (lane & 7)] != 0);
}

// A wave's part in staging a chunk: 64 quads of pixels, of one channel group or two.
struct Task {
  int at;           // in LDS, or kNowhere
  unsigned inside;  // which pixels lie in the image
  int c, off;       // first channel; where its first pixel lies there
};
constexpr int kNowhere = -1;
constexpr int kStaged = 0, kMultiplied = 1;

// What a wave asks for, and when: a tile's chunks one after the other, then the next tile's.
template <int WN>
struct Stage {
  Arguments arguments;
  const Work& work;
  const Places& at;
  const Shared& shared;
  u32x4* lds;
  __amdgpu_buffer_rsrc_t irsrc;
  int wave, lane, hw4;
  int tile = 0, chunk = 0;  // to ask for next
  int to, from;     // of the wave's part of a tile's chunks: place in LDS, or kNowhere; place of its first pixel in the input, in a chunk's first channel
  unsigned inside;  // which pixels lie in the image
  u32x4 x[8];
  float scale = 1.f;
  unsigned own_asides = 0;
  bool begins = false;  // what was asked for is a tile's first chunk
  int asked_tile = 0, asked_chunk = 0;
  int done = 0;         // chunks that the wave has multiplied
  bool unread = false;  // the tensor's first pixels, with columns outside of the image before them

  __device__ __forceinline__ bool more() const { return tile < work.tiles; }
  __device__ __forceinline__ void begin(int k) {
    tile = k;
    chunk = 0;
  }
  // one of 512 values from all over a tile's input, which tell what it has to be scaled by
  __device__ __forceinline__ unsigned sample(const Tile& t) const {
    const int hw = at.H * at.W, ch0 = work.c_beg * 8 * at.kgs, channels = min(work.rounds * 8 * at.kgs, at.C - ch0);
    const int pixel = max((int)(t.row0 - over(t.row0, at.m_ihs) * at.ihs) * at.sub - at.pad, 0) * at.W + (lane & 15) + t.staged * (wave >> 1);
    return __builtin_amdgcn_raw_buffer_load_b32(
        irsrc, 4 * ((int)over(t.q0, at.m_strips) * at.C * hw + min(pixel, hw - 1)) + (ch0 + (channels * (lane >> 4 | (wave & 1) << 2) >> 3)) * hw4, 0, 0);
  }
  __device__ __forceinline__ void keep_sample(int k, unsigned some) const {
    const unsigned most = wave_max(some & 0x7fffffff);
    if (lane == 0) shared.most[k % 3 * kWaves + wave] = most;
  }
  __device__ __forceinline__ Task task_of(int tile, int chunk, int lane) const {
    Task t;
    const Tile place = tile_of<WN>(arguments, work, tile);
    const unsigned n = wave * 64 + lane, kg = __umulhi(n, 0xffffffffu / (unsigned)place.staged + 1), quad = n - kg * place.staged;
    const bool exists = kg < (unsigned)at.kgs;
    t.at = exists ? (int)(kg * at.lpad + 4 * quad) : kNowhere;
    t.c = ((work.c_beg + chunk) * at.kgs + (exists ? (int)kg : 0)) * 8;
    t.off = source_of(at, place, quad, t.inside);
    if (!exists) {
      t.off = kNone;
      t.inside = 0;
    }
    return t;
  }
  // asks for the next chunk
  __device__ __forceinline__ void ask() {
    if (chunk == 0) {
      const Task t = task_of(tile, 0, lane);
      to = t.at;
      inside = t.inside;
      from = t.off + (t.c - work.c_beg * at.kgs * 8) * hw4;
      unread = __builtin_amdgcn_ballot_w64(t.off < 0) != 0;
    }
    begins = chunk == 0;
    asked_tile = tile;
    asked_chunk = chunk;
    const int c = (work.c_beg + chunk) * at.kgs * 8;
    if (c + at.kgs * 8 <= at.C) {
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = __builtin_amdgcn_raw_buffer_load_b128(irsrc, max(from + c * hw4, 0), j * hw4, 0);
    } else {  // channels that do not exist are zero
      const int kg = to < 0 ? 0 : (unsigned)to / (unsigned)at.lpad;
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = __builtin_amdgcn_raw_buffer_load_b128(irsrc, c + 8 * kg + j < at.C ? max(from + c * hw4, 0) + j * hw4 : kOutside, 0, 0);
    }
    if (++chunk == work.rounds) begin(tile + 1);
  }
  // the exponent bits of 2^e in the tile's scale, of a number that is not scaled yet (where it may underflow)
  __device__ __forceinline__ unsigned unscaled(int e) const { return (unsigned)min(max(2 * 127 + e - (int)(bits_of(scale) >> 23), 0), 255) << 23; }
  // Quads with inputs that the products cannot be formed of: listed, and zero in their parts.
  __device__ __forceinline__ void set_aside(int buf) {
    int lane = this->lane;  // (likewise)
    asm volatile("" : "+v"(lane));
    const Task task = task_of(asked_tile, asked_chunk, lane);
    const int plane = at.kgs * at.lpad, pixel = task.at < 0 ? 0 : task.at % at.lpad, slot = asked_tile % 3;
#pragma nounroll
    for (int e = 0; e < 4; ++e) {
      const bool exists = task.at >= 0 && task.inside >> e & 1;
      float v[8];
      unsigned which = 0;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        v[j] = float_of(__builtin_amdgcn_raw_buffer_load_b32(irsrc, exists && task.c + j < at.C ? task.off + 4 * e + (task.c + j) * hw4 : kOutside, 0, 0));
        const unsigned u = bits_of(v[j]) & 0x7fffffff;
        if (u - 1 < unscaled(kSmall2) - 1 || u >= unscaled(kLarge)) which |= 1u << j;
      }
      float kept[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) kept[j] = which >> j & 1 ? 0.f : v[j];
      u32x4 part[2];
      f16x2 zeros = {0, 0};
      cut2(kept, scale, part[0], part[1], zeros);
      if (task.at >= 0) {
        u32x4* d = lds + buf * plane + task.at + e;
        d[0] = part[0];
        d[kPart] = part[1];
      }
      while (const unsigned long long lanes = __builtin_amdgcn_ballot_w64(which != 0)) {
        const int j = __builtin_ctz(which | 256);
        float y = v[0];
#pragma unroll
        for (int q = 1; q < 8; ++q) y = j == q ? v[q] : y;
        const unsigned u = bits_of(y) & 0x7fffffff, n = own_asides + __builtin_amdgcn_mbcnt_hi(lanes >> 32, __builtin_amdgcn_mbcnt_lo(lanes, 0));
        const bool listed = u >= unscaled(kLeastListed) && u < unscaled(kMostListed);
        if (which && n < kMostAside) shared.aside[(slot * kWaves + wave) * kMostAside + n] = make_int2((task.c + j) << 10 | (pixel + e), (int)bits_of(y));
        own_asides = min(own_asides + (__builtin_amdgcn_ballot_w64(which && !listed) ? kNotListed : __builtin_popcountll(lanes)), kNotListed);
        which &= which - 1;
      }
    }
  }
  // cuts what was asked for into parts, in buffer `buf`
  __device__ __forceinline__ bool keep(int buf) {  // (true: set_aside is to follow)
    bool odd = false;
    // (unknown to the compiler until here, which else would wait for them and begin with them before the loop that this is in)
#pragma unroll
    for (int i = 0; i < 8; ++i) asm volatile("" : "+v"(x[i]));
    asm volatile("" : "+v"(inside));
    const int slot = asked_tile % 3;
    if (begins) {
      // Their largest is scaled to [2^11, 2^12).
      const unsigned most = wave_max(shared.most[slot * kWaves + (lane & 7)]);
      const int shift = most ? min(max(138 - (int)(most >> 23), -100), 100) : 6;
      scale = __builtin_bit_cast(float, (127 + shift) << 23);
      own_asides = 0;
      if (wave == 0) shared.shift[slot] = shift;
    }
    if (wave * 64 < at.kgs * (at.lpad >> 2)) {
      if (unread && asked_chunk == 0 && work.c_beg == 0) {  // read from the tensor's first pixel on instead of from before it
        for (int p = 0; p < 3; ++p)
#pragma unroll
          for (int i = 0; i < 8; ++i) x[i] = from + 4 * p < 0 ? u32x4{0, x[i][0], x[i][1], x[i][2]} : x[i];
      }
      f16x2 zeros = {0, 0};
      unsigned least = ~0u;  // of the inputs' bits without the sign, doubled, less one: zeros come out on top
      u32x4* d = lds + buf * at.kgs * at.lpad + to;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          v[i] = float_of(x[i][e]);
          least = min(least, (x[i][e] << 1) - 1);
        }
        u32x4 hi, lo;
        cut2(v, inside >> e & 1 ? scale : 0.f, hi, lo, zeros);
        if (to != kNowhere) {
          d[e] = hi;
          d[e + kPart] = lo;
        }
      }
      const bool infinite = __builtin_bit_cast(unsigned, zeros) & 0x7fff7fff;
      odd = __builtin_amdgcn_ballot_w64(infinite | (least < 2 * unscaled(kSmall2) - 1)) != 0;
    }
    return odd;
  }
  // how many inputs of a chunk are set aside (the count counts only once the tile's last chunk is staged)
  __device__ __forceinline__ void publish() const {
    const int slot = asked_tile % 3;
    if (begins) shared.asides[16 * slot + 8 + wave] = own_asides > kMostAside || (own_asides > 2 && own_asides * (unsigned)work.rounds > kMostAside);
    shared.asides[16 * slot + wave] = own_asides;
  }
  // A wave goes on as soon as what it needs is there, not when the last one has done all that it has to: it multiplies a chunk once all have
  // staged their part of it, and stages the next one once all have multiplied the one before, which the buffer held.
  __device__ __forceinline__ void arrive(int which) const {
    if (lane == 0) __hip_atomic_fetch_add(shared.counts + which, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  __device__ __forceinline__ void wait_for(int which, int chunks) const {
    for (int i = 0; i < 1 << 22; ++i) {  // (all waves are resident, and none waits for what comes after its own: the bound is never met)
      if (__builtin_amdgcn_readfirstlane(__hip_atomic_load(shared.counts + which, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP)) >= kWaves * chunks) break;
      __builtin_amdgcn_s_sleep(1);
    }
  }
};

constexpr int kInputs = 2;
constexpr int kSumPairs = 4;  // pairs of steps after which sums go to those that are rounded less often

// A tile's products.  In: the first chunk is staged, in buffer `buf`, and the first weights are asked for.  Out: the next tile's first chunk is
// staged, if there is one.
template <int NB, int WN>
__device__ __forceinline__ void multiply(Stage<WN>& stage, int k, unsigned some, const int* first, const u32x4* lds, const Weights& weights, Step (&ahead)[2], int base,
                                         const int (&bpos)[kTile], f32x16 (&sum)[2][kTile], int& buf) {
  const Places& at = stage.at;
  const int plane = at.kgs * at.lpad;
  const unsigned tap_bits = at.ks > 4 ? 3 : 2, kg_bits = 7 - 2 * tap_bits;
  // where a step's input is read: the blocks in the two halves of a lane's registers
  auto place_of = [&](unsigned word, int r) {
    return buf * plane + (int)(__builtin_amdgcn_ubfe(word, 16 + 8 * r, tap_bits) + __umul24(__builtin_amdgcn_ubfe(word, 16 + 8 * r + tap_bits, tap_bits), at.wp) +
                               __umul24(__builtin_amdgcn_ubfe(word, 16 + 8 * r + 2 * tap_bits, kg_bits), at.lpad));
  };
  int place[2];
  struct Input { u32x4 v[2][2]; };
  Input input[kInputs];
  auto read = [&](Input& in, int b) {
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      in.v[r][0] = lds[place[r] + bpos[b]];
      in.v[r][1] = lds[place[r] + bpos[b] + kPart];
    }
  };
  int next_step = base + 2;
  // a step's products, while the input of the block after is read; `reads`: of the next step's first block as well
  auto step = [&](Step& now, const Step& next, auto turn, bool reads) {
    constexpr int kFirst = NB * decltype(turn)::value % kInputs;
    const unsigned word = now.word;
    const u32x4 near = now.p[0], off = now.p[1];
    const u32x4 far = __builtin_bit_cast(u32x4, __builtin_bit_cast(f16x8, near) * (f16x8)(_Float16)(1 / kRest));
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const Input& in = input[(kFirst + b) % kInputs];
      if (b + 1 < NB) {
        read(input[(kFirst + b + 1) % kInputs], b + 1);
      } else if (reads) {
        place[0] = place_of(next.word, 0);
        place[1] = place_of(next.word, 1);
        read(input[(kFirst + NB) % kInputs], 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      sum[0][b] = product<true>(off, in.v[0][0], in.v[1][0], (int)word, sum[0][b]);
      sum[0][b] = product<true>(near, in.v[0][0], in.v[1][0], (int)word, sum[0][b]);
      sum[0][b] = product<true>(far, in.v[0][1], in.v[1][1], (int)word, sum[0][b]);
      __builtin_amdgcn_sched_barrier(0);
    }
    fetch(weights, next_step++, now);
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr std::integral_constant<int, 0> even;
  constexpr std::integral_constant<int, 1> odd;
  int since = 0;
  int from = first[0];
  for (int round = 0; round < stage.work.rounds; ++round) {
    const int to = first[round + 1], pairs = (to - from) >> 1;
    from = to;
    const bool stages = stage.more();
    place[0] = place_of(ahead[0].word, 0);
    place[1] = place_of(ahead[0].word, 1);
    read(input[0], 0);
    if (stages) stage.ask();
    __builtin_amdgcn_sched_barrier(0);
    // (Two steps by themselves, in which what is staged next is on its way: the loop's waits would include it.)
    step(ahead[0], ahead[1], even, true);
    step(ahead[1], ahead[0], odd, pairs > 1);
    const int when = (stage.wave < kWaves / 2 ? pairs : 2 * pairs) / 3;  // (the two waves of a SIMD not at the same time)
    bool odd_inputs = false;
    for (int i = 1;; ++i) {
      if (++since >= kSumPairs) {
        since = 0;
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int k = 0; k < 16; ++k) {
            sum[1][b][k] += sum[0][b][k];
            sum[0][b][k] = 0.f;
          }
      }
      if (i == max(when, 1) && stages) {
        stage.wait_for(kMultiplied, stage.done);
        odd_inputs = stage.keep(buf ^ 1);
        if (!odd_inputs) {
          stage.publish();
          stage.arrive(kStaged);
        }
      }
      if (i >= pairs) break;
      step(ahead[0], ahead[1], even, true);
      step(ahead[1], ahead[0], odd, i + 1 < pairs);
    }
    if (stages) {
      if (__builtin_expect(odd_inputs, 0)) {
        stage.set_aside(buf ^ 1);
        stage.publish();
        stage.arrive(kStaged);
      }
      if (round + 1 == stage.work.rounds && k + 2 < stage.work.tiles) stage.keep_sample(k + 2, some);
      stage.arrive(kMultiplied);
      stage.wait_for(kStaged, ++stage.done);
    }
    buf ^= 1;
  }
}

// What is added to a tile's sums with FMAs: few tiles have any.  `sums`: room for a block of them, per wave.
template <int WM, int WN>
__device__ __forceinline__ void add_singles(Arguments arguments, const Work& work, const Places& at, const Shared& shared, const Tile& tile, const Own& own_blocks, int block, int slot,
                                            unsigned long long listed, const int (&bpos)[kTile], f32x16 (&sum)[2][kTile], float* sums, int wave, int lane) {
  asm volatile("" : "+v"(lane));  // (unknown to the compiler, which else would keep much of this in registers all the while)
  const auto& g = arguments->g;
  const auto& w = arguments->w;
  const int wm = wave % WM, wn = wave / WM, oc0 = (work.mt * WM + wm) * 32, loose = w.loose_count[block], shift = shared.shift[slot];
  const float scale = __builtin_bit_cast(float, (127 + shift) << 23);
  const __amdgpu_buffer_rsrc_t irsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(arguments->in), 0, g.in_bytes, 0x00020000);
  // inputs set aside are added in the order of their places: sums do not depend on who came first
  const int2 own = listed >> lane & 1 ? shared.aside[slot * kWaves * kMostAside + lane] : make_int2(0x7fffffff, 0);
  int before = 0;
  for (unsigned long long left = listed; left; left &= left - 1) before += __builtin_amdgcn_readlane(own.x, __builtin_ctzll(left)) < own.x;
#pragma unroll
  for (int b = 0; b < kTile; ++b) {
    if (b >= own_blocks.count) break;
#pragma unroll
    for (int i = 0; i < 16; ++i) sums[i * 64 + lane] = sum[0][b][i];
    const Pixel p = pixel_of<WN>(at, work, tile, wn * tile.count + own_blocks.first + b, lane);
    // weights that fp16 parts do not hold
#pragma nounroll
    for (int e = 0; e < loose; ++e) {
      const int where = w.loose[kMostLoose * block + e].x, row = where & 31, r = where >> 5 & 7, s = where >> 8 & 7, c = where >> 11;
      const float weight = __builtin_bit_cast(float, w.loose[kMostLoose * block + e].y);
      const int chunk = c / (8 * at.kgs);
      if (chunk < work.c_beg || chunk >= work.c_beg + work.rounds) continue;
      const int iy = (int)(p.oy * at.stride + r) * at.sub - at.pad, ix = (int)(p.w * at.stride + s) * at.sub - at.pad;
      const bool inside = iy >= 0 && iy < at.H && ix >= 0 && ix < at.W && p.n < (unsigned)at.N && (lane >> 5) == (row >> 2 & 1);
      const float v = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                          irsrc, inside ? 4 * (int)(((p.n * at.C + c) * at.H + iy) * at.W + ix) : kOutside, 0, 0)) * scale;
      float& to = sums[((row >> 3) * 4 + (row & 3)) * 64 + lane];
      to = fmaf(v, weight, to);
    }
    // inputs set aside, with the weights that are not among those
    const int cpad = 8 * at.kgs * g.chunks;
#pragma nounroll
    for (int e = 0; e < __builtin_popcountll(listed); ++e) {
      const int who = __builtin_ctzll(__builtin_amdgcn_ballot_w64(before == e));
      const int where = __builtin_amdgcn_readlane(own.x, who), c = where >> 10;
      const float v = float_of(__builtin_amdgcn_readlane(own.y, who)) * scale;
      int tap = -1;  // of the lane's pixel that reads it
      for (int r = 0; r < at.ks; ++r) {
        const int s = (where & 1023) - bpos[b] - r * at.wp;
        if (s >= 0 && s < at.ks) tap = r * at.ks + s;
      }
      if (!__builtin_amdgcn_ballot_w64(tap >= 0)) continue;
#pragma nounroll
      for (int i = 0; i < 16; i += 8) {  // (eight at a time: the trips to memory are what this costs)
        float weight[8];
        int exponent[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int row = 2 * i + 8 * (j / 4) + 4 * (lane >> 5) + j % 4, oc = oc0 + row;
          weight[j] = tap >= 0 && oc < g.K ? w.dense[((size_t)oc * at.ks * at.ks + tap) * cpad + c] : 0.f;
          exponent[j] = w.row_exp[block * 32 + row];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float scaled = ldexpf(weight[j], -exponent[j]);
          sums[(i + j) * 64 + lane] = fmaf(v, fabsf(scaled) >= kLeast ? scaled : 0.f, sums[(i + j) * 64 + lane]);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) sum[0][b][i] = sums[i * 64 + lane];
  }
}

// Returns which tiles are to be computed again.
template <int WM, int WN>
__device__ __forceinline__ unsigned long long multiply_all(Arguments arguments, const Work& work, const Places& at, const Shared& shared, u32x4* lds, int wave, int lane) {
  const auto& g = arguments->g;
  const auto& w = arguments->w;
  const int wm = wave % WM, wn = wave / WM, oc0 = (work.mt * WM + wm) * 32, block = min(work.mt * WM + wm, g.mblocks - 1);
  const int* const first = w.first + block * g.chunks + work.c_beg;
  const int base = first[0];
  const Weights weights = {__builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(w.steps), 0, w.step_bytes, 0x00020000), lane};
  float* const sums = shared.sums + wave * 1024;
  Stage<WN> stage{arguments, work, at, shared, lds, __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(arguments->in), 0, g.in_bytes, 0x00020000), wave, lane, 4 * g.H * g.W};
  unsigned some_first[2] = {stage.sample(tile_of<WN>(arguments, work, 0)), 0};
  if (work.tiles > 1) some_first[1] = stage.sample(tile_of<WN>(arguments, work, 1));
  stage.ask();
  unsigned long long again = 0;
  Step ahead[2];
  auto first_weights = [&]() {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      fetch(weights, base + i, ahead[i]);
      __builtin_amdgcn_sched_barrier(0);  // in this order: the loop waits for the first set only
    }
  };
  first_weights();
  int buf = 0;
  stage.keep_sample(0, some_first[0]);
  if (work.tiles > 1) stage.keep_sample(1, some_first[1]);
  if (wave == 0 && lane < 2) shared.counts[lane] = 0;
  __syncthreads();
  if (stage.keep(0)) stage.set_aside(0);
  stage.publish();
  __syncthreads();
  for (int k = 0; k < work.tiles; ++k) {
    const int slot = k % 3;
    asm volatile("" : "+v"(lane));
    unsigned some = 0;
    if (k + 2 < work.tiles) {
      some = stage.sample(tile_of<WN>(arguments, work, k + 2));
    }
    if (too_many_soon(shared, slot, lane)) {  // what is left of it is not staged
      again |= 1ull << k;
      if (k + 2 < work.tiles) stage.keep_sample(k + 2, some);
      __syncthreads();
      if (stage.tile == k || work.rounds == 1) stage.begin(k + 1);
      if (stage.more()) {
        stage.ask();
        if (stage.keep(buf ^ 1)) stage.set_aside(buf ^ 1);
        stage.publish();
        stage.arrive(kStaged);
        stage.arrive(kMultiplied);
        ++stage.done;
      }
      __syncthreads();
      buf ^= 1;
      continue;
    }
    const Tile tile = tile_of<WN>(arguments, work, k);
    const Own own = own_of(work, tile, k, wave);
    int bpos[kTile];
    f32x16 sum[2][kTile];
#pragma unroll
    for (int b = 0; b < kTile; ++b) {
      bpos[b] = lds_of(at, tile, pixel_of<WN>(at, work, tile, wn * tile.count + own.first + min(b, own.count - 1), lane));
#pragma unroll
      for (int i = 0; i < 16; ++i) sum[0][b][i] = sum[1][b][i] = 0.f;
    }
    if constexpr (kTile == 4) {
      if (own.count == 4) multiply<4>(stage, k, some, first, lds, weights, ahead, base, bpos, sum, buf);
    }
    if (own.count == 2) multiply<2>(stage, k, some, first, lds, weights, ahead, base, bpos, sum, buf);
    else if (own.count == 3) multiply<3>(stage, k, some, first, lds, weights, ahead, base, bpos, sum, buf);
    first_weights();
    if (too_many(shared, slot, lane)) {
      again |= 1ull << k;
      continue;
    }
#pragma unroll
    for (int b = 0; b < kTile; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) sum[0][b][i] += sum[1][b][i];
    const unsigned listed = shared.asides[16 * slot + lane / kMostAside];  // by the wave whose list this lane may read
    const unsigned long long some_listed = __builtin_amdgcn_ballot_w64(lane % kMostAside < listed);
    if (some_listed || w.loose_count[block])
      add_singles<WM, WN>(arguments, work, at, shared, tile, own, block, slot, some_listed, bpos, sum, sums, wave, lane);
    const Stores stores = stores_of(arguments, work, oc0);
    const int shift = shared.shift[slot];
    int4 e[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) e[i] = *reinterpret_cast<const int4*>(w.row_exp + block * 32 + 8 * i + 4 * (lane >> 5));
    int unknown = lane;  // (likewise)
    asm volatile("" : "+v"(unknown));
#pragma unroll
    for (int b = 0; b < kTile; ++b) {
      if (!(own.stores >> b & 1)) continue;
      const int out = out_of(arguments, pixel_of<WN>(at, work, tile, wn * tile.count + own.first + b, unknown), unknown);
#pragma unroll
      for (int i = 0; i < 16; i += 4) {
        float v[4];
        v[0] = ldexpf(sum[0][b][i], e[i / 4].x - shift);
        v[1] = ldexpf(sum[0][b][i + 1], e[i / 4].y - shift);
        v[2] = ldexpf(sum[0][b][i + 2], e[i / 4].z - shift);
        v[3] = ldexpf(sum[0][b][i + 3], e[i / 4].w - shift);
        store(stores, unknown, i, out, v);
      }
    }
  }
  return again;
}

// A tile with bf16 parts, which hold every number, by all waves: inputs that cannot be written as fp16 ones, or weights.  A wave with a sum that is
// not finite computes its outputs with FMAs.  Both are here to be right; latency bounds them.
template <int WM, int WN>
__device__ __forceinline__ void compute_again(Arguments arguments, const Work& work, const Places& at, const Shared& shared, u32x4* lds, int k, int wave_id, int lane) {
  constexpr int NB = kTile;
  const auto& g = arguments->g;
  const auto& w = arguments->w;
  const Tile tile = tile_of<WN>(arguments, work, k);
  const __amdgpu_buffer_rsrc_t irsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(arguments->in), 0, g.in_bytes, 0x00020000);
  const int hw4 = 4 * g.H * g.W, plane = at.kgs * at.lpad;
  const int wave = wave_id, wm = wave % WM, wn = wave / WM, block = min(work.mt * WM + wm, g.mblocks - 1), oc0 = (work.mt * WM + wm) * 32;
  const Own own = own_of(work, tile, k, wave);
  f32x16 sum[2][NB];
  int bpos[NB], out[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const bool exists = own.stores >> b & 1;
    const Pixel p = pixel_of<WN>(at, work, tile, wn * tile.count + own.first + min(b, own.count - 1), lane);
    bpos[b] = lds_of(at, tile, p);
    out[b] = exists ? out_of(arguments, p, lane) : kOutside;
#pragma unroll
    for (int i = 0; i < 16; ++i) sum[0][b][i] = sum[1][b][i] = 0.f;
  }
  const unsigned tap_bits = at.ks > 4 ? 3 : 2, kg_bits = 7 - 2 * tap_bits;
  const __amdgpu_buffer_rsrc_t wrsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(w.steps), 0, w.step_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t srsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(w.slots), 0, w.step_bytes / kBytes * kSlotBytes, 0x00020000);
  int next_step = w.first[block * g.chunks + work.c_beg];
  struct { u32x4 v[2]; unsigned word; } ahead;
  auto fetch_slots = [&](int step) {
    ahead.v[0] = __builtin_amdgcn_raw_buffer_load_b128(srsrc, lane * 16, step * kSlotBytes, 0);
    ahead.v[1] = __builtin_amdgcn_raw_buffer_load_b128(srsrc, lane * 16 + 1024, step * kSlotBytes, 0);
    ahead.word = __builtin_amdgcn_raw_buffer_load_b32(wrsrc, lane * 4 + 2048, step * kBytes, 0);
  };
  fetch_slots(next_step);
  const int end = w.first[block * g.chunks + work.c_beg + work.rounds];
  for (int round = 0; round < work.rounds; ++round) {
    __syncthreads();
    for (int task = wave_id * 64 + lane; task < at.kgs * tile.staged; task += 512) {
      const int kg = task / tile.staged, quad = task - kg * tile.staged, c = ((work.c_beg + round) * at.kgs + kg) * 8;
      unsigned inside;
      const int from = source_of(at, tile, quad, inside) + c * hw4;
      u32x4 x[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = __builtin_amdgcn_raw_buffer_load_b128(irsrc, c + j < at.C ? max(from, 0) + j * hw4 : kOutside, 0, 0);
      for (int p = 0; p < 3; ++p)  // (read from the tensor's first pixel on instead of from before it)
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = from + 4 * p < 0 ? u32x4{0, x[j][0], x[j][1], x[j][2]} : x[j];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = inside >> e & 1 ? float_of(x[j][e]) : 0.f;
        u32x4 part[3];
        cut(v, part[0], part[1], part[2]);
#pragma unroll
        for (int p = 0; p < 3; ++p) lds[p * plane + kg * at.lpad + 4 * quad + e] = part[p];
      }
    }
    __syncthreads();
    for (bool last = false; !last && next_step < end;) {
      const u32x4 w0 = ahead.v[0], w1 = ahead.v[1];
      const unsigned word = ahead.word;
      fetch_slots(++next_step);  // (none behind the last: zeros)
      last = __builtin_amdgcn_readfirstlane(word) >> 31;
      int place[2];
#pragma unroll
      for (int r = 0; r < 2; ++r)
        place[r] = (int)(__builtin_amdgcn_ubfe(word, 16 + 8 * r, tap_bits) + __umul24(__builtin_amdgcn_ubfe(word, 16 + 8 * r + tap_bits, tap_bits), at.wp) +
                         __umul24(__builtin_amdgcn_ubfe(word, 16 + 8 * r + 2 * tap_bits, kg_bits), at.lpad));
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = float_of(j < 4 ? w0[j % 4] : w1[j % 4]);
      u32x4 a[3];
      cut(v, a[0], a[1], a[2]);
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        u32x4 in[2][3];
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
          for (int p = 0; p < 3; ++p) in[r][p] = lds[place[r] + bpos[b] + p * plane];
        // all products but low times low, smallest first
        constexpr int pa[8] = {2, 1, 2, 1, 0, 1, 0, 0}, pb[8] = {1, 2, 0, 1, 2, 0, 1, 0};
#pragma unroll
        for (int t = 0; t < 8; ++t) sum[t < 7][b] = product<false>(a[pa[t]], in[0][pb[t]], in[1][pb[t]], (int)word, sum[t < 7][b]);
      }
    }
  }
  const Stores stores = stores_of(arguments, work, oc0);
  float odd = 0;  // NaN once a sum is infinite or NaN
#pragma unroll
  for (int i = 0; i < 16; i += 4)
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[j] = sum[0][b][i + j] + sum[1][b][i + j];
        odd = fmaf(v[j], 0.f, odd);
        v[j] *= kUnscale;
      }
      store(stores, lane, i, out[b], v);
    }
  if (__ballot(odd != 0.f) == 0) return;
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): what follows stores over what was stored, by other lanes
  const int ch0 = work.c_beg * 8 * g.kgs, ch1 = min(g.C, (work.c_beg + work.rounds) * 8 * g.kgs), cpad = 8 * g.kgs * g.chunks;
#pragma nounroll
  for (int b = 0; b < own.count; ++b) {
    if (!(own.stores >> b & 1)) continue;
    const Pixel p = pixel_of<WN>(at, work, tile, wn * tile.count + own.first + b, lane);
    float sums[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) sums[i] = 0;
#pragma nounroll
    for (int c = ch0; c < ch1; c += 8)
#pragma nounroll
      for (int r = 0; r < g.ks; ++r)
#pragma nounroll
        for (int s = 0; s < g.ks; ++s) {
          const int iy = (int)(p.oy * g.stride + r) * g.sub - g.pad, ix = (int)(p.w * g.stride + s) * g.sub - g.pad;
          const bool inside = iy >= 0 && iy < g.H && ix >= 0 && ix < g.W && p.n < (unsigned)g.N;
          float v[8];
#pragma unroll
          for (int q = 0; q < 8; ++q)
            v[q] = float_of(__builtin_amdgcn_raw_buffer_load_b32(irsrc, inside && c + q < g.C ? 4 * (int)(((p.n * g.C + c + q) * g.H + iy) * g.W + ix) : kOutside, 0, 0));
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int oc = oc0 + 8 * (i / 4) + 4 * (lane >> 5) + i % 4;
            const u32x4* d = reinterpret_cast<const u32x4*>(w.dense + (((size_t)min(oc, g.K - 1) * g.ks + r) * g.ks + s) * cpad + c);
            const u32x4 d0 = d[0], d1 = d[1];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
              const float f = float_of(q < 4 ? d0[q % 4] : d1[q % 4]);
              if (f != 0.f) sums[i] = fmaf(v[q], f, sums[i]);
            }
          }
        }
    const int to = out_of(arguments, p, lane);
#pragma unroll
    for (int i = 0; i < 16; i += 4) {
      float v[4] = {sums[i], sums[i + 1], sums[i + 2], sums[i + 3]};
      store(stores, lane, i, to, v);
    }
  }
}

template <int WM, int WN>
__global__ __launch_bounds__(512, 2) void relay_kernel(const MatArguments) {
  static_assert(WM * WN == kWaves);
  extern __shared__ u32x4 lds[];  // [parts][buffers][kgs][lpad], then Shared
  Arguments arguments = (Arguments)__builtin_amdgcn_kernarg_segment_ptr();
  const auto& g = arguments->g;
  const auto& w = arguments->w;
  if ((int)((blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3)) >= g.runs * g.mtiles * g.csplit) return;
  const int lane = threadIdx.x & 63, wave_id = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const Work work = work_of(arguments);
  const Places at = places_of(arguments);
  const Shared shared = shared_of(arguments, lds);
  unsigned long long again = 0;
  if (w.loose_count[0] < 0) {  // (so of all blocks: the filter's weights cannot be written in parts)
    again = work.tiles == 64 ? ~0ull : (1ull << work.tiles) - 1;
  } else {
    again = multiply_all<WM, WN>(arguments, work, at, shared, lds, wave_id, lane);
  }
  while (again) {
    compute_again<WM, WN>(arguments, work, at, shared, lds, __builtin_ctzll(again), wave_id, lane);
    again &= again - 1;
  }
}

template <int WM, int WN>
int launch_one(const MatGeom& g, const float* d_in, float* d_out, const MatWeights& weights, hipStream_t stream) {
  auto kern = relay_kernel<WM, WN>;
  static std::atomic<bool> lds_set{false};  // per instantiation; setting the attribute twice is harmless
  if (!lds_set.load(std::memory_order_acquire)) {
    TETRIS_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kMatLds));
    lds_set.store(true, std::memory_order_release);
  }
  const int grid = 8 * ceil_div(g.runs * g.mtiles * g.csplit, 8);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(512), mat_lds_bytes(g), stream, MatArguments{d_in, d_out, weights, g});
  TETRIS_HIP(hipGetLastError());
  return TETRIS_OK;
}

}  // namespace

int launch_relay(const MatGeom& g, const float* d_in, float* d_out, const MatWeights& weights, int relu, hipStream_t stream) {
  MatGeom k = g;
  k.relu = relu;
  k.quads = stores_quads(g, d_out);
  const MatShape& c = kMatShapes[g.cfg];
  if (c.wm == 8) return launch_one<8, 1>(k, d_in, d_out, weights, stream);
  if (c.wm == 4) return launch_one<4, 2>(k, d_in, d_out, weights, stream);
  if (c.wm == 2) return launch_one<2, 4>(k, d_in, d_out, weights, stream);
  return fail(TETRIS_EINVAL, "no matrix kernel of configuration %d", g.cfg);
}

}  // namespace tetris
