// kf_prior_conv.hpp — the convolution kernels of the prior's training step.
//
// A wavefront keeps its share of a layer's weights in registers (144 of them) as
// the A operand of v_mfma_f32_16x16x32_bf16 and takes 16 pixels at a time as the B
// operand, sixteen bytes of eight channels per lane and step (no im2col matrix).  With
// the weights as A, a lane
// holds output channels of one pixel; their order over the tiles is chosen so that
// a lane's channels are contiguous and it stores them as whole vectors.  Each output
// is one MFMA chain over k = 0, 32, ... from zero, the sequence of prior_infer_fused, so
// the two give the same bits.
#pragma once

#include "kf_prior_net.hpp"

namespace kf {

constexpr int kConvThreads = 256;
constexpr int kConvWaves = kConvThreads / kWave;

// Output channel of row i (0..15) of A tile t when a wave has NT tiles: lane q = i / 4
// then holds channels 4 NT q .. 4 NT q + 4 NT - 1 over its NT accumulators.
template <int NT>
__device__ __forceinline__ int tile_channel(int t, int i) {
  return (i >> 2) * 4 * NT + 4 * t + (i & 3);
}

// The 16 bytes at element `at` of a map, element 0 if not `in`.  The offset goes through an
// opaque register: otherwise the compiler sees that the value will not be used, and
// branches around each load.
__device__ __forceinline__ uint4 load_vec(const uint16_t* p, bool in, int at) {
  return *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(p) + opaque_u32(in ? 2u * (unsigned)at : 0u));
}

// Stores N (a multiple of 4) BF16 values, two in a word, to p (8-byte aligned; 16-byte
// aligned when N is a multiple of 8).
template <int N>
__device__ __forceinline__ void store_words(uint16_t* p, const uint32_t* w) {
  if constexpr (N % 8 == 0) {
#pragma unroll
    for (int i = 0; i < N / 2; i += 4) *reinterpret_cast<uint4*>(p + 2 * i) = make_uint4(w[i], w[i + 1], w[i + 2], w[i + 3]);
  } else {
#pragma unroll
    for (int i = 0; i < N / 2; i += 2) *reinterpret_cast<uint2*>(p + 2 * i) = make_uint2(w[i], w[i + 1]);
  }
}
// The same from floats, rounded to nearest even.
template <int N>
__device__ __forceinline__ void store_bf16(uint16_t* p, const float* v) {
  uint32_t w[N / 2];
#pragma unroll
  for (int i = 0; i < N / 2; ++i) w[i] = pack_bf16(v[2 * i], v[2 * i + 1]);
  store_words<N>(p, w);
}

// The same, and (bits not NULL) which of the N (8 or 16) stored values are positive, value
// i in bit i: all that the backward pass needs of them under a ReLU, in a sixteenth of
// the bytes.
template <int N>
__device__ __forceinline__ void store_bf16_signs(uint16_t* p, uint8_t* bits, const float* v) {
  typedef short s2 __attribute__((ext_vector_type(2)));
  typedef unsigned short u2 __attribute__((ext_vector_type(2)));
  uint32_t w[N / 2], m = 0;
#pragma unroll
  for (int i = 0; i < N / 2; ++i) w[i] = pack_bf16(v[2 * i], v[2 * i + 1]);
  store_words<N>(p, w);
  if (!bits) return;  // uniform
#pragma unroll
  for (int i = 0; i < N / 2; ++i) {
    const s2 pos = __builtin_elementwise_max(__builtin_bit_cast(s2, w[i]), (s2){0, 0});
    const u2 one = __builtin_elementwise_min(__builtin_bit_cast(u2, pos), (u2){1, 1});
    m |= __builtin_bit_cast(uint32_t, one) << 2 * i;  // value 2 i in bit 2 i, 2 i + 1 in bit 16 + 2 i
  }
  m |= m >> 15;
  if constexpr (N == 8)
    *bits = (uint8_t)m;
  else
    *reinterpret_cast<uint16_t*>(bits) = (uint16_t)m;
}

// v of the lane above in its row of 16, `edge` in the row's last lane.
__device__ __forceinline__ uint4 lane_above(uint4 v, uint4 edge) {
  auto mv = [](uint32_t e, uint32_t x) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)e, (int)x, 0x101, 0xf, 0xf, false);
  };
  return make_uint4(mv(edge.x, v.x), mv(edge.y, v.y), mv(edge.z, v.z), mv(edge.w, v.w));
}

// The 16-pixel tiles of wave group `unit` of `units` in a block, of `blocks` blocks: first,
// first + step, ... below last.  Blocks go to the eight XCDs (each with its own L2) in
// turn, and neighbouring tiles read the same rows, so each XCD takes a run of them.
struct TileRun {
  int first, last, step;
  __device__ __forceinline__ TileRun(int tiles, int block, int blocks, int unit, int units) {
    if (blocks % 8 == 0) {
      const int x = block % 8;
      first = (int)((long)tiles * x / 8) + block / 8 * units + unit;
      last = (int)((long)tiles * (x + 1) / 8);
      step = blocks / 8 * units;
    } else {
      first = block * units + unit;
      last = tiles;
      step = blocks * units;
    }
  }
};

// Layer 1 forward: a block makes four output rows of one sample.  The nine input rows
// of both planes are staged in LDS as BF16 pairs (previous, current), so that one
// 32-bit LDS read is one tap's two channels.
constexpr int kL1Rows = 4;                      // output rows of a block
constexpr int kL1In = 2 * kL1Rows + 1;          // input rows under them
constexpr int kL1Pitch = kW0 + 4;               // columns -1 .. 159 from 3 on
static_assert(kConv[0].hout % kL1Rows == 0, "layer-1 row groups");

// One operand tile of layer 1's weights (WeightCopies::w1), its 18 columns padded to 32.
__device__ __forceinline__ uint4 conv1_weights(const uint16_t* W1, int t, int r, int q) {
  return *reinterpret_cast<const uint4*>(W1 + operand_at(kConv[0].cout, tile_channel<2>(t, r), 8 * q));
}

// Bound by the map's stores (79 MB at batch 256).  A row of the patch is loaded as 16-byte
// vectors of both frames and written as whole vectors (column 0 at 4, so that they are
// aligned; column -1 at 3 is always outside the frame).  Batch 256: 22.5 us; with single pixels,
// two divisions each, and the weights as 16-bit loads 31.
__global__ __launch_bounds__(kConvThreads) void conv1_forward(const float* frames, const int32_t* pairs,
                                                              const uint16_t* W1, const float* bias, uint16_t* Yb,
                                                              uint8_t* signs) {
  constexpr ConvShape c = kConv[0];
  typedef float f4 __attribute__((ext_vector_type(4), aligned(4)));
  __shared__ __align__(16) uint32_t patch[kL1In][kL1Pitch];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, q = lane >> 4;
  const int n = blockIdx.y, oy0 = blockIdx.x * kL1Rows;
  const float* f0 = frames + (long)pairs[2 * n] * (kH0 * kW0);
  const float* f1 = frames + (long)pairs[2 * n + 1] * (kH0 * kW0);
  constexpr int V = kW0 / 4, E = kL1In * V, PER = (E + kConvThreads - 1) / kConvThreads;
  f4 v[PER][2];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int e = threadIdx.x + kConvThreads * u, o = (2 * oy0 - 1) * kW0 + 4 * e;  // row 2 oy0 - 1 + e / V
    v[u][0] = v[u][1] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    if (e < E && o >= 0) {
      v[u][0] = *reinterpret_cast<const f4*>(f0 + o);
      v[u][1] = *reinterpret_cast<const f4*>(f1 + o);
    }
  }
  uint4 w[2];
  float b[8];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    w[t] = conv1_weights(W1, t, r, q);
#pragma unroll
    for (int j = 0; j < 4; ++j) b[4 * t + j] = bias[8 * q + 4 * t + j];
  }
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int e = threadIdx.x + kConvThreads * u;
    if (e < E)
      *reinterpret_cast<uint4*>(&patch[e / V][4 + 4 * (e % V)]) =
          make_uint4(pack_bf16(v[u][0].x, v[u][1].x), pack_bf16(v[u][0].y, v[u][1].y), pack_bf16(v[u][0].z, v[u][1].z),
                     pack_bf16(v[u][0].w, v[u][1].w));
  }
  if (threadIdx.x < kL1In) patch[threadIdx.x][3] = 0u;
  int off[4];  // the lane's four taps (4 q ..), tap 8 standing in for those past the kernel
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int tap = min(4 * q + e, 8);
    off[e] = (tap / 3) * kL1Pitch + tap % 3 + 3;
  }
  __syncthreads();
  const uint32_t* flat = &patch[0][0];
  for (int tile = wave; tile < kL1Rows * c.wout / 16; tile += kConvWaves) {
    const int p = tile * 16 + r, oy = p / c.wout, ox = p - oy * c.wout;
    const int at = 2 * oy * kL1Pitch + 2 * ox;
    uint32_t v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = flat[at + off[e]];
      if (4 * q + e > 8) v[e] = 0u;
    }
    const uint4 a = make_uint4(v[0], v[1], v[2], v[3]);
    float y[8];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
      acc = mfma32(w[t], a, acc);
#pragma unroll
      for (int j = 0; j < 4; ++j) y[4 * t + j] = fmaxf(acc[j] + b[4 * t + j], 0.0f);
    }
    const long o = (((long)n * c.hout + oy0 + oy) * c.wout + ox) * c.cout + 8 * q;
    store_bf16_signs<8>(Yb + o, signs ? signs + o / 8 : nullptr, y);
  }
}

// The operand tile of 16 pixels of layer L's forward: the rows of input pixels under them,
// a wavefront's own in LDS.  The map is read as it lies in memory (a pixel's two columns 2 ox
// and 2 ox + 1 are 2 cin channels on end: a quarter wave touches two lines, where operands
// loaded straight from the map touch sixteen, and the L1's lookups bound the kernel), and
// the tile's left neighbour once.  Column 2 ox - 1 is the pixel before's second one.  A
// pixel's 16-byte chunks are permuted by its index so that the operand reads' eight
// pixels at a time meet no bank twice.
template <int L>
struct ConvTile {
  static constexpr ConvShape c = kConv[L];
  static constexpr int PC = c.cin / 8, U = 2 * PC;      // chunks of an input pixel, of an output pixel's two columns
  static constexpr int PER = 16 * U / kWave;            // loads of an input row
  static constexpr int kChunks = 3 * (16 * U + PC);     // LDS of a wave: three rows, and the pixels left of them
  static_assert(U == 8 || U == 16, "32 or 64 input channels");
  uint4 v[3][PER], left;
  bool in[3][PER], left_in;

  static __device__ __forceinline__ int chunk(int pixel, int i) { return pixel * U + (i ^ (U == 8 ? pixel >> 1 : pixel)); }
  static __device__ __forceinline__ bool row_in(int oy, int ky) {
    const int iy = 2 * oy + ky - 1;
    return iy >= 0 && (2 * c.hout <= c.hin || iy < c.hin);
  }

  __device__ __forceinline__ void load(const uint16_t* X, int tile, int M, int lane) {
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int e = u * kWave + lane, i = e % U;
      const int m = min(tile * 16 + e / U, M - 1);
      const int n = m / (c.hout * c.wout), p = m - n * (c.hout * c.wout), oy = p / c.wout, ox = p - oy * c.wout;
      const int at = ((n * c.hin + 2 * oy - 1) * c.win + 2 * ox) * c.cin + 8 * i;
#pragma unroll
      for (int ky = 0; ky < 3; ++ky) {
        in[ky][u] = row_in(oy, ky);
        v[ky][u] = load_vec(X, in[ky][u], at + ky * c.win * c.cin);
      }
    }
    const int m = tile * 16, ky = lane / PC;
    const int n = m / (c.hout * c.wout), p = m - n * (c.hout * c.wout), oy = p / c.wout, ox = p - oy * c.wout;
    left = make_uint4(0u, 0u, 0u, 0u);
    if (lane < 3 * PC && ox > 0 && row_in(oy, ky))
      left = *reinterpret_cast<const uint4*>(X + ((n * c.hin + 2 * oy - 1 + ky) * c.win + 2 * ox - 1) * c.cin + 8 * (lane % PC));
  }

  __device__ __forceinline__ void stage(uint4* lds, int lane) {
#pragma unroll
    for (int ky = 0; ky < 3; ++ky)
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int e = u * kWave + lane;
        lds[ky * 16 * U + chunk(e / U, e % U)] = in[ky][u] ? v[ky][u] : make_uint4(0u, 0u, 0u, 0u);
      }
    if (lane < 3 * PC) lds[3 * 16 * U + lane] = left;
  }

  // The operand of tap (ky, kx) and channels 32 k .. of pixel r, chunk q of four; ox: its column.
  static __device__ __forceinline__ uint4 operand(const uint4* lds, int ky, int kx, int k, int r, int q, int ox) {
    if (kx > 0) return lds[ky * 16 * U + chunk(r, (kx - 1) * PC + 4 * k + q)];
    const uint4 a = lds[r > 0 ? ky * 16 * U + chunk(r - 1, PC + 4 * k + q) : 3 * 16 * U + ky * PC + 4 * k + q];
    return ox > 0 ? a : make_uint4(0u, 0u, 0u, 0u);
  }
};

// Layers 2-4 forward.  NT: 16-channel tiles of a wave (COUT / (16 NT) waves cover a
// pixel's channels), chosen so that every layer's share is 144 weight registers (two
// waves per SIMD); F32: FP32 output (layer 4, which the pooling reads), else BF16.  The
// next tile's loads are in flight while this one is multiplied.  Bound by memory (layer 2
// at batch 256: 120 MB).  Batch 256: layers 2 / 3 / 4 in 26 / 18 / 13 us (with weight rows on
// end: 27 / 23 / 17; operands straight from the map, the left column from the neighbouring
// lane: 27 / 27 / 20; all nine from the map: 32 / 33 / 23; GEMMs staged through LDS took
// 570 us with layer 1's 30).
template <int L, int NT, bool F32>
__global__ __launch_bounds__(kConvThreads, 2) void conv_forward(const uint16_t* X, const uint16_t* W, const float* bias,
                                                                uint16_t* Yb, float* Y, uint8_t* signs, int M) {
  constexpr ConvShape c = kConv[L];
  using T = ConvTile<L>;
  constexpr int KS = c.kc / 32, CS = c.cin / 32, GROUPS = c.cout / (16 * NT);
  static_assert(2 * c.wout == c.win && c.kc == 9 * c.cin && c.cin % 32 == 0, "layer shape");
  __shared__ uint4 s_in[kConvWaves][T::kChunks];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, q = lane >> 4;
  const int group = wave % GROUPS, ch0 = group * 16 * NT;
  const TileRun run((M + 15) / 16, blockIdx.x, gridDim.x, wave / GROUPS, kConvWaves / GROUPS);
  T in;
  if (run.first < run.last) in.load(X, run.first, M, lane);
  uint4 w[KS][NT];
  float b[4 * NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
#pragma unroll
    for (int s = 0; s < KS; ++s)
      w[s][t] = *reinterpret_cast<const uint4*>(W + operand_at(c.cout, ch0 + tile_channel<NT>(t, r), 32 * s + 8 * q));
#pragma unroll
    for (int j = 0; j < 4; ++j) b[4 * t + j] = bias[ch0 + 4 * NT * q + 4 * t + j];
  }
  uint4* lds = s_in[wave];
  for (int tile = run.first; tile < run.last; tile += run.step) {
    in.stage(lds, lane);
    if (tile + run.step < run.last) in.load(X, tile + run.step, M, lane);
    wave_lds_sync();
    const int m = min(tile * 16 + r, M - 1);  // rows past the end repeat the last one
    const int ox = m % c.wout;
    v4f acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const uint4 a = T::operand(lds, s / CS / 3, s / CS % 3, s % CS, r, q, ox);
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = mfma32(w[s][t], a, acc[t]);
    }
    wave_lds_sync();
    if (tile * 16 + r >= M) continue;
    float y[4 * NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) y[4 * t + j] = fmaxf(acc[t][j] + b[4 * t + j], 0.0f);
    const long o = (long)m * c.cout + ch0 + 4 * NT * q;
    if constexpr (F32) {
#pragma unroll
      for (int i = 0; i < 4 * NT; i += 4) *reinterpret_cast<float4*>(Y + o + i) = make_float4(y[i], y[i + 1], y[i + 2], y[i + 3]);
    } else {
      store_bf16_signs<4 * NT>(Yb + o, signs ? signs + o / 8 : nullptr, y);
    }
  }
}

// Weight gradients contract over pixels, while the maps keep a pixel's channels
// together.  The tiles are staged in LDS as they lie in memory, one row of channels per
// pixel, and the operands come from transposing LDS reads (ds_read_b64_tr_b16): of
// each 16-lane group, lanes 4 i .. 4 i + 3 address the 16 channels of pixel row i, and
// lane c receives channel c of the four rows.  A fragment is two such reads, pixels
// 4 q .. 4 q + 3 and 16 + 4 q .. of the 32 staged (both operands in the same order).
// Row pitches are odd multiples of 8 dwords, so that the eight rows of 32 bytes that
// a half-wave reads cover all 64 banks.
constexpr int kWgradStep = 32;  // pixels (or samples) staged at a time
typedef short v4s __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4s lds_v4s;

__device__ __forceinline__ uint4 transposed_fragment(const uint16_t* rows, int pitch, int c0, int r, int q) {
  const uint16_t* p = rows + (4 * q + (r >> 2)) * pitch + c0 + 4 * (r & 3);
  const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(p));
  const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(p + 16 * pitch));
  const uint2 a = __builtin_bit_cast(uint2, lo), b = __builtin_bit_cast(uint2, hi);
  return make_uint4(a.x, a.y, b.x, b.y);
}

// Layer 1's weight gradient, taken where layer 2's input gradient makes layer 1's output
// gradient, which then never goes to memory: dW1[co][k] = sum_m dY1[m][co] col[m][k], col
// the im2col element of the two frames.  A wave's tile is 8 x 2 2x2 blocks; it holds the
// 9 x 33 input pixels under them as BF16 pairs (previous, current) in LDS, writes its
// gradients there row by row of the blocks, and makes the 32 x 18 products of 32 pixels
// from transposing reads of the gradients and 16-bit reads of the pairs.  The gradient
// (79 MB at batch 256) was written by one launch and read by another: layer 2's backward
// pass 74 us and 31 more, now 66 for both.
struct Conv1Grad {
  const float* frames;
  const int32_t* pairs;
  float* part;  // a plane per block
};
constexpr int kC1Pitch = 36;                        // pairs of a row: column -1 at 3, columns 0 .. 31 from 4 (16-byte aligned)
constexpr int kC1Patch = 9 * kC1Pitch;              // pairs of a wave
constexpr int kC1DyPitch = 32 + 16;                 // gradients of a pixel, bank-spreading
constexpr int kC1Wave = 2 * kC1Patch + kWgradStep * kC1DyPitch;  // a wave's LDS, in 16-bit elements
static_assert(kC1Wave % 8 == 0 && kC1Patch % 4 == 0, "16-byte alignment");

struct Conv1GradWave {
  uint32_t* patch;
  uint16_t* dy;
  int base[2];  // of the lane's column of the 16-column tiles, in 16-bit elements
  v4f acc[2][2];

  __device__ __forceinline__ Conv1GradWave(uint16_t* lds, int lane) {
    patch = reinterpret_cast<uint32_t*>(lds);
    dy = lds + 2 * kC1Patch;
    const int r = lane & 15, q = lane >> 4;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int k = min(16 * t + r, kConv[0].kc - 1), tap = k >> 1;  // columns past the kernel are not kept
      base[t] = 2 * ((4 * (q >> 1) + tap / 3) * kC1Pitch + 16 * (q & 1) + tap % 3 + 3) + (k & 1);
#pragma unroll
      for (int c = 0; c < 2; ++c) acc[c][t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }

  // The input pixels of rows 8 jt - 1 .. 8 jt + 7 and columns 32 it - 1 .. 32 it + 31 of
  // sample n (0 outside the frames): 72 vectors of four columns and nine pixels left of
  // them.  The loads are issued by load(), the pairs go to LDS in stage().
  typedef float f4 __attribute__((ext_vector_type(4), aligned(4)));
  f4 v[2][2];
  __device__ __forceinline__ void load(const Conv1Grad& g, int lane, int n, int jt, int it) {
    const float* f[2] = {g.frames + (long)g.pairs[2 * n] * (kH0 * kW0), g.frames + (long)g.pairs[2 * n + 1] * (kH0 * kW0)};
    const int y0 = 8 * jt - 1, y1 = lane < 8 ? y0 + 8 : y0 + lane - 8;
    const int at = (y0 + (lane >> 3)) * kW0 + 32 * it + 4 * (lane & 7);
    const int left = y1 * kW0 + 32 * it - 1, last = y1 * kW0 + 32 * it + 4 * lane;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      v[0][c] = v[1][c] = f4{0.0f, 0.0f, 0.0f, 0.0f};
      if (at >= 0) v[0][c] = *reinterpret_cast<const f4*>(f[c] + at);
      if (lane < 8)
        v[1][c] = *reinterpret_cast<const f4*>(f[c] + last);
      else if (lane < 17 && y1 >= 0 && it > 0)
        v[1][c].x = f[c][left];
    }
  }
  __device__ __forceinline__ void stage(int lane) {
    uint32_t w[2][4];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) w[u][e] = pack_bf16(v[u][0][e], v[u][1][e]);
    *reinterpret_cast<uint4*>(patch + (lane >> 3) * kC1Pitch + 4 + 4 * (lane & 7)) = make_uint4(w[0][0], w[0][1], w[0][2], w[0][3]);
    if (lane < 8)
      *reinterpret_cast<uint4*>(patch + 8 * kC1Pitch + 4 + 4 * lane) = make_uint4(w[1][0], w[1][1], w[1][2], w[1][3]);
    else if (lane < 17)
      patch[(lane - 8) * kC1Pitch + 3] = w[1][0];
  }

  // The products of pixel row py of the blocks: dy holds its pixels px = 0, then px = 1.
  __device__ __forceinline__ void add_row(int lane, int py) {
    const int r = lane & 15, q = lane >> 4;
    const uint16_t* pairs = reinterpret_cast<const uint16_t*>(patch);
    uint4 a[2], b[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) a[c] = transposed_fragment(dy, kC1DyPitch, 16 * c, r, q);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      uint32_t w[4];  // pixels 4 q .. 4 q + 3 of px = 0, then of px = 1, as the fragments order them
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint16_t* p = pairs + base[t] + 4 * py * kC1Pitch + 4 * (i >> 1) + 16 * (i & 1);
        w[i] = (uint32_t)p[0] | (uint32_t)p[8] << 16;
      }
      b[t] = make_uint4(w[0], w[1], w[2], w[3]);
    }
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int t = 0; t < 2; ++t) acc[c][t] = mfma32(a[c], b[t], acc[c][t]);
  }

  // The block's plane: the sum over its waves, in order.  s: kConvWaves 1024 floats.
  __device__ __forceinline__ void finish(const Conv1Grad& g, int block, float* s) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, q = lane >> 4;
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) s[wave * 1024 + (16 * c + 4 * q + j) * 32 + 16 * t + r] = acc[c][t][j];
    __syncthreads();
    constexpr int kc = kConv[0].kc;
    for (int e = threadIdx.x; e < kConv[0].cout * kc; e += kConvThreads) {
      const int i = e / kc * 32 + e % kc;
      float v = s[i];
#pragma unroll
      for (int u = 1; u < kConvWaves; ++u) v = v + s[u * 1024 + i];
      g.part[(long)block * (kConv[0].cout * kc) + e] = v;
    }
  }
};

// Input gradient of layer L (1..3), ReLU mask of the layer below and that layer's bias
// sums in one pass: dX[n][iy][ix][ci] = sum over the taps (ky, kx) that reach the
// pixel, in that order, of sum_co dY[n][oy][ox][co] W[co][(ky, kx, ci)]; 0 where the
// forward map is not positive (its signs, one bit a value).  A wave takes 16 2x2 pixel blocks (rows 2j, 2j + 1,
// columns 2i, 2i + 1): with stride 2 their nine taps read only the four output pixels
// (j .. j + 1, i .. i + 1), so dY is read four times and every product is needed.
// The weights (per tap an operand copy with rows ci) stay in 144 registers.
// Each tap's product is an MFMA chain of its own from zero and the taps are added in
// FP32: the bits of a column-gradient GEMM followed by col2im, without the FP32 column
// matrix (354 MB for layer 2 at batch 256).  bpart: per block and channel the FP32 sum
// of the unrounded gradients.  Layer 2's output stays on the chip (Conv1Grad).  Bound by
// memory: with the forward map in place of its signs (layer 2 at batch 256: 79 MB) the
// three layers' backward passes took 160 us instead of 140; the GEMM, col2im, conversion and column sums took 4.3 ms.
// Block `block` of `blocks`; s_b: kDgradLds floats of LDS.
template <int L>
struct DgradShape {
  static constexpr int NT = L == 3 ? 1 : 2;                // 16-channel tiles of a wave
  static constexpr int GROUPS = kConv[L].cin / (16 * NT);  // waves that cover a pixel's channels
};
constexpr int kDgradLds = kConvWaves * 32;

template <int L>
__device__ __forceinline__ void dgrad_block(const uint16_t* dY, const uint16_t* Wt, const uint8_t* signs, uint16_t* dX,
                                            float* bpart, int M, int block, int blocks, float* s_sum,
                                            const Conv1Grad& g, uint16_t* lds) {
  constexpr ConvShape c = kConv[L];
  constexpr int NT = DgradShape<L>::NT, KS = c.cout / 32, GROUPS = DgradShape<L>::GROUPS, CH = 4 * NT;
  static_assert(c.win == 2 * c.wout && (c.hin == 2 * c.hout || c.hin == 2 * c.hout - 1) && kConvWaves % GROUPS == 0,
                "layer shape");
  float (*s_b)[16 * NT] = reinterpret_cast<float (*)[16 * NT]>(s_sum);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, q = lane >> 4;
  const int gw = block * kConvWaves + wave, group = gw % GROUPS;
  const int ch0 = group * 16 * NT;
  uint4 w[9][KS][NT];
#pragma unroll
  for (int tap = 0; tap < 9; ++tap)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int s = 0; s < KS; ++s)
        w[tap][s][t] = *reinterpret_cast<const uint4*>(Wt + tap * c.cin * c.cout +
                                                       operand_at(c.cin, ch0 + tile_channel<NT>(t, r), 32 * s + 8 * q));
  float bs[CH];
#pragma unroll
  for (int j = 0; j < CH; ++j) bs[j] = 0.0f;
  const TileRun run((M + 15) / 16, block, blocks, wave / GROUPS, kConvWaves / GROUPS);
  [[maybe_unused]] Conv1GradWave first(lds + wave * kC1Wave, lane);
  for (int tile = run.first; tile < run.last; tile += run.step) {
    bool live = true;
    int m, n, j, i;
    if constexpr (L == 1) {  // 8 x 2 blocks, 75 tiles of a sample
      static_assert(c.wout % 8 == 0 && c.hout % 2 == 0, "layer shape");
      const int at = __builtin_amdgcn_readfirstlane(tile);
      n = at / (c.hout * c.wout / 16);
      const int t = at - n * (c.hout * c.wout / 16), jt = t / (c.wout / 8), it = t - jt * (c.wout / 8);
      j = 2 * jt + (r >> 3);
      i = 8 * it + (r & 7);
      m = (n * c.hout + j) * c.wout + i;
      first.load(g, lane, n, jt, it);
    } else {
      live = tile * 16 + r < M;
      m = live ? tile * 16 + r : M - 1;
      n = m / (c.hout * c.wout);
      const int p = m - n * (c.hout * c.wout);
      j = p / c.wout;
      i = p - j * c.wout;
    }
    // the four pixels' sign bits of the lane's channels
    uint32_t sign[2][2];
    int out[2][2];
#pragma unroll
    for (int py = 0; py < 2; ++py)
#pragma unroll
      for (int px = 0; px < 2; ++px) {
        const int iy = min(2 * j + py, c.hin - 1), ix = 2 * i + px;
        out[py][px] = ((n * c.hin + iy) * c.win + ix) * c.cin + ch0 + CH * q;
        sign[py][px] = (uint32_t)signs[(unsigned)out[py][px] / 8u] >> (out[py][px] & 4);
      }
    uint4 a[2][2][KS];  // dY at (j + dj, i + di), 0 outside the map
    // (the column to the right is the next lane's, but for the last pixel of the tile's row)
    constexpr int kEnd = L == 1 ? 7 : 15;
#pragma unroll
    for (int dj = 0; dj < 2; ++dj) {
      const bool in = dj == 0 || j + 1 < c.hout;
      const uint16_t* src = dY + (in ? (m + dj * c.wout) * c.cout : 0) + 8 * q;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        a[dj][0][s] = load_vec(dY, in, (m + dj * c.wout) * c.cout + 8 * q + 32 * s);
        a[dj][1][s] = make_uint4(0u, 0u, 0u, 0u);
        if ((r & kEnd) == kEnd && in && i + 1 < c.wout) a[dj][1][s] = *reinterpret_cast<const uint4*>(src + c.cout + 32 * s);
      }
    }
#pragma unroll
    for (int dj = 0; dj < 2; ++dj)
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        // (selects only here: before, each would wait for its load)
        if (dj == 1 && j + 1 >= c.hout) a[dj][0][s] = make_uint4(0u, 0u, 0u, 0u);
        const uint4 own = a[dj][1][s];
        uint4 v = lane_above(a[dj][0][s], own);
        if (i + 1 >= c.wout) v = make_uint4(0u, 0u, 0u, 0u);
        if (kEnd < 15 && (r & kEnd) == kEnd) v = own;
        a[dj][1][s] = v;
      }
    if constexpr (L == 1) first.stage(lane);
#pragma unroll
    for (int py = 0; py < 2; ++py) {
#pragma unroll
      for (int px = 0; px < 2; ++px) {
        float sum[CH];
#pragma unroll
        for (int e = 0; e < CH; ++e) sum[e] = 0.0f;
#pragma unroll
        for (int ky = 1 - py; ky < 3; ky += 2)
#pragma unroll
          for (int kx = 1 - px; kx < 3; kx += 2) {
            const int dj = ky == 0 ? 1 : 0, di = kx == 0 ? 1 : 0;  // odd pixels: tap 0 is the next output pixel, tap 2 this one
#pragma unroll
            for (int t = 0; t < NT; ++t) {
              v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
              for (int s = 0; s < KS; ++s) acc = mfma32(w[ky * 3 + kx][s][t], a[dj][di][s], acc);
#pragma unroll
              for (int e = 0; e < 4; ++e) sum[4 * t + e] = sum[4 * t + e] + acc[e];
            }
          }
        if (live && (c.hin == 2 * c.hout || 2 * j + py < c.hin)) {
#pragma unroll
          for (int e = 0; e < CH; ++e) {
            const int keep = (int)(sign[py][px] << (31 - e)) >> 31;  // 0 or all ones
            sum[e] = __int_as_float(__float_as_int(sum[e]) & keep);
            bs[e] = bs[e] + sum[e];
          }
          if constexpr (L == 1)
            store_bf16<CH>(first.dy + (16 * px + r) * kC1DyPitch + CH * q, sum);
          else
            store_bf16<CH>(dX + out[py][px], sum);
        }
      }
      if constexpr (L == 1) {
        wave_lds_sync();
        first.add_row(lane, py);
        wave_lds_sync();
      }
    }
  }
#pragma unroll
  for (int e = 0; e < CH; ++e) {
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) bs[e] = bs[e] + __shfl_xor(bs[e], o, kWave);
    if (r == 0) s_b[wave][CH * q + e] = bs[e];
  }
  __syncthreads();
  if (threadIdx.x < c.cin) {
    const int g = threadIdx.x / (16 * NT), k = threadIdx.x - g * 16 * NT;
    float v = s_b[g][k];
    for (int u = g + GROUPS; u < kConvWaves; u += GROUPS) v = v + s_b[u][k];
    bpart[(long)block * c.cin + threadIdx.x] = v;
  }
  if constexpr (L == 1) first.finish(g, block, reinterpret_cast<float*>(lds));
}

// Weight gradients of the fully connected layers, dW5[j][c] = sum_n dH[n][j] X5[n][c] and
// dW6[t][k] = sum_n dO[n][t] H[n][k], and the loss mean((O - T)^2): five blocks of their
// own beside layer 2's backward pass, which they finish long before (a launch of their
// own would cost its 4 us, blocks in the final sums 13 us at batch 256).
constexpr int kX5Pitch = 144;  // row of pooled features and twist, rounded up to MFMA tiles
constexpr int kDoPitch = 16;   // row of output gradients, rounded up to an MFMA tile
constexpr int kFcBlocks = 5;   // four of 64 rows of dW5, one of dW6 and the loss
struct FcGradArgs {
  const uint16_t *X5b, *Hb, *dOb, *dHb;
  const float *O, *target;
  float *dW5, *dW6, *loss;
  int batch;
};

// Columns i0 .. of A (WA of them, rows of PA elements) against B's rows of PB: wave w
// makes row tile w / WPT and column tiles (w % WPT) NT .. of C[i][k] = sum_n A[n][i]
// B[n][k], 32 samples a step, the next step's vectors in flight.
template <int PA, int WA, int PB, int NT, int WPT>
__device__ __forceinline__ void fc_weight_gradient(const uint16_t* A, int i0, const uint16_t* B, int batch, int rows,
                                                   int cols, float* out, uint16_t* s) {
  constexpr int pa = WA + 16 + (WA / 16 % 2) * 16, pb = PB + 16 + (PB / 16 % 2) * 16;
  static_assert(pa / 16 % 2 == 1 && pb / 16 % 2 == 1, "bank-spreading pitches");
  constexpr int VA = kWgradStep * WA / 8, VB = kWgradStep * PB / 8, PER = (VA + VB + kConvThreads - 1) / kConvThreads;
  uint16_t* sa = s;
  uint16_t* sb = s + kWgradStep * pa;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, q = lane >> 4;
  const int it = wave / WPT * 16, k0 = wave % WPT * NT * 16;
  v4f acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  uint4 v[PER];
  auto place = [&](int u, bool& isa, int& row, int& col) {  // where vector u of this thread lies; false: it has none
    const int e = threadIdx.x + kConvThreads * u;
    isa = e < VA;
    const int f = isa ? e : e - VA, per = isa ? WA / 8 : PB / 8;
    row = f / per;
    col = 8 * (f - row * per);
    return e < VA + VB;
  };
  auto load = [&](int n0) {
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      bool isa;
      int row, col;
      v[u] = make_uint4(0u, 0u, 0u, 0u);
      if (place(u, isa, row, col) && n0 + row < batch)
        v[u] = *reinterpret_cast<const uint4*>(isa ? A + (long)(n0 + row) * PA + i0 + col : B + (long)(n0 + row) * PB + col);
    }
  };
  load(0);
  for (int n0 = 0; n0 < batch; n0 += kWgradStep) {
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      bool isa;
      int row, col;
      if (place(u, isa, row, col)) *reinterpret_cast<uint4*>((isa ? sa : sb) + row * (isa ? pa : pb) + col) = v[u];
    }
    if (n0 + kWgradStep < batch) load(n0 + kWgradStep);
    __syncthreads();
    const uint4 a = transposed_fragment(sa, pa, it, r, q);
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = mfma32(a, transposed_fragment(sb, pb, k0 + 16 * t, r, q), acc[t]);
    __syncthreads();
  }
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int i = i0 + it + 4 * q + j, k = k0 + 16 * t + r;
      if (i < rows && k < cols) out[i * cols + k] = acc[t][j];
    }
}

// Block b < kFcBlocks of the above; s: kFcLds elements of LDS (dW6's tiles, the larger).
constexpr int kFcLds = kWgradStep * (kDoPitch + 32 + kHidden + 16);
static_assert(kFcLds >= kWgradStep * (64 + 16 + kX5Pitch + 32), "dW5's tiles");
__device__ __forceinline__ void fc_block(const FcGradArgs& a, int b, uint16_t* s) {
  if (b + 1 < kFcBlocks) {
    fc_weight_gradient<kHidden, 64, kX5Pitch, kX5Pitch / 16, 1>(a.dHb, 64 * b, a.X5b, a.batch, kHidden, kFc1In, a.dW5, s);
    return;
  }
  fc_weight_gradient<kDoPitch, kDoPitch, kHidden, kHidden / 16 / kConvWaves, kConvWaves>(a.dOb, 0, a.Hb, a.batch, kTwist,
                                                                                         kHidden, a.dW6, s);
  float* red = reinterpret_cast<float*>(s);
  const int n = a.batch * kTwist, tid = threadIdx.x;
  float v = 0.0f;
  for (int i = tid; i < n; i += kConvThreads) {
    const float d = a.O[i] - a.target[i];
    v = v + d * d;
  }
  red[tid] = v;
  __syncthreads();
  for (int o = kConvThreads / 2; o > 0; o >>= 1) {
    if (tid < o) red[tid] += red[tid + o];
    __syncthreads();
  }
  if (tid == 0 && a.loss) *a.loss = red[0] * (1.0f / (float)n);
}

// Weight gradient of layer L (1..3): dW[co][k] = sum_m dY[m][co] col[m][k], col the
// im2col element read straight from the map X.  A block takes one split of the pixels
// and COB output channels; a wave 2 x 9 tiles of them, so that eleven fragment reads
// feed eighteen MFMAs.  Per step of 32 pixels the next step's vectors are in flight
// while this one's tiles are multiplied.  Each split writes its own plane
// (reduce_parts adds them in order).  Bound by the L1 path of the map
// loads and the LDS reads.  Batch 256: layers 2 / 3 / 4 in 45 / 24 / 15 us (250 / 240 /
// 198 TFLOP/s); the im2col matrices and the GEMMs over them took 2.3 ms with layer 1.
template <int L>
struct WgradShape {
  static constexpr int COB = L == 1 ? 64 : 32;             // output channels of a block
  static constexpr int GROUPS = kConv[L].cout / COB;
  static constexpr int NW = kConv[L].kc / (9 * 16);        // waves along the weight columns
  static constexpr int kColPitch = kConv[L].kc + 16, kDyPitch = COB + 16;
  static constexpr int kColLds = kWgradStep * kColPitch, kDyLds = kWgradStep * kDyPitch;
  static_assert(NW * (COB / 32) == kConvWaves && kConv[L].kc % (9 * 16) == 0, "wave tiles");
};

// Block `block`; s_col: kColLds elements, s_dy: kDyLds.
template <int L>
__device__ __forceinline__ void wgrad_block(const uint16_t* dY, const uint16_t* X, float* part, int M, int steps_per_split,
                                            int block, uint16_t* s_col, uint16_t* s_dy) {
  constexpr ConvShape c = kConv[L];
  constexpr int COB = WgradShape<L>::COB, GROUPS = WgradShape<L>::GROUPS, NW = WgradShape<L>::NW;
  constexpr int kColPitch = WgradShape<L>::kColPitch, kDyPitch = WgradShape<L>::kDyPitch;
  constexpr int kTapVecs = c.cin / 8, kVecs = c.kc / 8, kPer = (kVecs + 7) / 8;  // eight threads per pixel
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, q = lane >> 4;
  // the groups of a split read the same map: keep them on one XCD (blocks go round-robin)
  const int b = block, split = b / (8 * GROUPS) * 8 + b % 8, group = b / 8 % GROUPS;
  const int co0 = group * COB;
  const int px = tid >> 3, v0 = tid & 7;
  const int first = split * steps_per_split, last = min(first + steps_per_split, (M + kWgradStep - 1) / kWgradStep);
  uint4 vc[kPer], vd;
  bool in[kPer], in_dy;  // vectors outside the map (zeroed when staged: a select here would wait for the load)
  auto load = [&](int step) {
    const int m = step * kWgradStep + px;
    const bool live = m < M;
    const int mm = live ? m : 0;
    const int n = mm / (c.hout * c.wout), p = mm - n * (c.hout * c.wout);
    const int oy = p / c.wout, ox = p - oy * c.wout;
    const int at = ((n * c.hin + 2 * oy - 1) * c.win + 2 * ox - 1) * c.cin;
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int v = v0 + 8 * u, tap = v / kTapVecs, ci = 8 * (v - tap * kTapVecs);
      const int ky = tap / 3, kx = tap - 3 * ky;
      const int iy = 2 * oy + ky - 1, ix = 2 * ox + kx - 1;
      in[u] = live && v < kVecs && iy >= 0 && iy < c.hin && ix >= 0;
      vc[u] = load_vec(X, in[u], at + (ky * c.win + kx) * c.cin + ci);
    }
    in_dy = live && v0 < COB / 8;
    vd = load_vec(dY, in_dy, m * c.cout + co0 + 8 * v0);
  };
  v4f acc[2][9];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int i = 0; i < 9; ++i) acc[t][i] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  const int cw = wave / NW * 32, nw = wave % NW * (9 * 16);  // the wave's first channel and column
  if (first < last) load(first);
  for (int step = first; step < last; ++step) {
#pragma unroll
    for (int u = 0; u < kPer; ++u)
      if (v0 + 8 * u < kVecs) *reinterpret_cast<uint4*>(&s_col[px * kColPitch + 8 * (v0 + 8 * u)]) =
            in[u] ? vc[u] : make_uint4(0u, 0u, 0u, 0u);
    if (v0 < COB / 8) *reinterpret_cast<uint4*>(&s_dy[px * kDyPitch + 8 * v0]) = in_dy ? vd : make_uint4(0u, 0u, 0u, 0u);
    __syncthreads();
    if (step + 1 < last) load(step + 1);
    uint4 a[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) a[t] = transposed_fragment(s_dy, kDyPitch, cw + 16 * t, r, q);
#pragma unroll
    for (int i = 0; i < 9; ++i) {
      const uint4 f = transposed_fragment(s_col, kColPitch, nw + 16 * i, r, q);
#pragma unroll
      for (int t = 0; t < 2; ++t) acc[t][i] = mfma32(a[t], f, acc[t][i]);
    }
    __syncthreads();
  }
  float* plane = part + (long)split * (c.cout * c.kc);
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int i = 0; i < 9; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) plane[(co0 + cw + 16 * t + 4 * q + j) * c.kc + nw + 16 * i + r] = acc[t][i][j];
}

// The backward pass of layer L: its weight gradient (blocks below wblocks), its input
// gradient (dblocks more) and, beside layer L = 1, the fully connected layers' blocks.
// Neither needs the other, and neither fills the chip at small batches: one launch
// instead of two.  Batch 256: layers 2 (with layer 1's weight gradient) / 3 / 4 in 59 / 33 /
// 21 us (in launches apart 126 / 58 / 42).
struct ConvBackArgs {
  const uint16_t *dY, *X, *Wt;
  const uint8_t* signs;  // of X
  uint16_t* dX;
  float *wpart, *bpart;
  int M, steps_per_split, wblocks, dblocks;
  FcGradArgs fc;
  Conv1Grad first;
};

template <int L>
__global__ __launch_bounds__(kConvThreads, 2) void conv_backward(ConvBackArgs a) {
  using S = WgradShape<L>;
  constexpr int kCol = L == 1 && kFcLds > S::kColLds ? kFcLds : S::kColLds;
  __shared__ __align__(16) uint16_t s_col[kCol], s_dy[S::kDyLds];
  static_assert(sizeof(s_dy) >= kDgradLds * sizeof(float) && kCol >= kConvWaves * (L == 1 ? kC1Wave : 0) &&
                    sizeof(s_col) >= (L == 1 ? kConvWaves * 1024 * sizeof(float) : 0),
                "LDS of the input gradient");
  const int b = blockIdx.x;  // every branch is uniform
  if (b < a.wblocks)
    wgrad_block<L>(a.dY, a.X, a.wpart, a.M, a.steps_per_split, b, s_col, s_dy);
  else if (b < a.wblocks + a.dblocks)
    dgrad_block<L>(a.dY, a.Wt, a.signs, a.dX, a.bpart, a.M, b - a.wblocks, a.dblocks, reinterpret_cast<float*>(s_dy), a.first,
                   s_col);
  else if constexpr (L == 1)
    fc_block(a.fc, b - a.wblocks - a.dblocks, s_col);
}

}  // namespace kf
