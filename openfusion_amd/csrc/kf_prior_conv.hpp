// kf_prior_conv.hpp — the convolution kernels of the prior's training step.
//
// A wavefront keeps its share of a layer's weights in registers (144 of them) as
// the A operand of v_mfma_f32_16x16x32_bf16 and takes 16 pixels at a time as the B
// operand, one 16-byte load of eight channels per lane and step straight from the
// NHWC BF16 map (through L1 / L2, no im2col matrix).  With the weights as A, a lane
// holds output channels of one pixel; their order over the tiles is chosen so that
// a lane's channels are contiguous and it stores them as whole vectors.  Each output
// is one MFMA chain over k = 0, 32, ... from zero, the sequence of gemm_bf16 and
// prior_infer_fused, so the three give the same bits.
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

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  return (uint32_t)bf16_rne(lo) | ((uint32_t)bf16_rne(hi) << 16);
}

// Stores N (a multiple of 4) floats as BF16 to p (8-byte aligned; 16-byte aligned when N is a multiple of 8).
template <int N>
__device__ __forceinline__ void store_bf16(uint16_t* p, const float* v) {
  if constexpr (N % 8 == 0) {
#pragma unroll
    for (int i = 0; i < N; i += 8)
      *reinterpret_cast<uint4*>(p + i) = make_uint4(pack_bf16(v[i], v[i + 1]), pack_bf16(v[i + 2], v[i + 3]),
                                                    pack_bf16(v[i + 4], v[i + 5]), pack_bf16(v[i + 6], v[i + 7]));
  } else {
#pragma unroll
    for (int i = 0; i < N; i += 4)
      *reinterpret_cast<uint2*>(p + i) = make_uint2(pack_bf16(v[i], v[i + 1]), pack_bf16(v[i + 2], v[i + 3]));
  }
}

// Layer 1 forward: a block makes four output rows of one sample.  The nine input rows
// of both planes are staged in LDS as BF16 pairs (previous, current), so that one
// 32-bit LDS read is one tap's two channels.
constexpr int kL1Rows = 4;                      // output rows of a block
constexpr int kL1In = 2 * kL1Rows + 1;          // input rows under them
constexpr int kL1Pitch = kW0 + 2;               // columns -1 .. 159 (and one of padding)
static_assert(kConv[0].hout % kL1Rows == 0, "layer-1 row groups");

// The input rows under output rows oy0 .. oy0 + kL1Rows - 1 (zero outside the frame).
__device__ __forceinline__ void stage_l1(uint32_t (*patch)[kL1Pitch], const float* f0, const float* f1, int oy0) {
  constexpr int E = kL1In * kL1Pitch, PER = (E + kConvThreads - 1) / kConvThreads;
  float v[PER][2];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int e = threadIdx.x + kConvThreads * u;
    const int row = e / kL1Pitch, col = e - row * kL1Pitch;
    const int iy = 2 * oy0 - 1 + row, ix = col - 1;
    const bool in = e < E && iy >= 0 && iy < kH0 && ix >= 0 && ix < kW0;
    const int o = in ? iy * kW0 + ix : 0;
    v[u][0] = in ? f0[o] : 0.0f;
    v[u][1] = in ? f1[o] : 0.0f;
  }
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int e = threadIdx.x + kConvThreads * u;
    if (e < E) patch[e / kL1Pitch][e % kL1Pitch] = pack_bf16(v[u][0], v[u][1]);
  }
}

__global__ __launch_bounds__(kConvThreads) void conv1_forward(const float* frames, const int32_t* pairs,
                                                              const uint16_t* W, const float* bias, uint16_t* Yb) {
  constexpr ConvShape c = kConv[0];
  __shared__ uint32_t patch[kL1In][kL1Pitch];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, q = lane >> 4;
  const int n = blockIdx.y, oy0 = blockIdx.x * kL1Rows;
  stage_l1(patch, frames + (long)pairs[2 * n] * (kH0 * kW0), frames + (long)pairs[2 * n + 1] * (kH0 * kW0), oy0);
  uint4 w[2];
  float b[8];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    uint16_t e[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) e[j] = 8 * q + j < c.kc ? W[tile_channel<2>(t, r) * c.kc + 8 * q + j] : (uint16_t)0;
    __builtin_memcpy(&w[t], e, 16);
#pragma unroll
    for (int j = 0; j < 4; ++j) b[4 * t + j] = bias[8 * q + 4 * t + j];
  }
  int off[4];  // the lane's four taps (4 q ..), tap 8 standing in for those past the kernel
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int tap = min(4 * q + e, 8);
    off[e] = (tap / 3) * kL1Pitch + tap % 3;
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
    store_bf16<8>(Yb + (((long)n * c.hout + oy0 + oy) * c.wout + ox) * c.cout + 8 * q, y);
  }
}

// Layers 2-4 forward.  Bound by the L1 path of the pixel loads (each map vector is read
// by up to four taps).  NT is chosen so that every layer's share is 144 weight
// registers (two waves per SIMD).  Batch 256: 31 / 33 / 23 us for layers 2 / 3 / 4
// (365 / 172 / 131 TFLOP/s), layer 1 30 us; GEMMs staged through LDS took 570 us for the
// four.  NT: 16-channel tiles of a wave (COUT / (16 NT) waves cover a
// pixel's channels); F32: FP32 output (layer 4, which the pooling reads), else BF16.
template <int L, int NT, bool F32>
__global__ __launch_bounds__(kConvThreads, 2) void conv_forward(const uint16_t* X, const uint16_t* W, const float* bias,
                                                                uint16_t* Yb, float* Y, int M) {
  constexpr ConvShape c = kConv[L];
  constexpr int KS = c.kc / 32, GROUPS = c.cout / (16 * NT);
  static_assert(2 * c.wout == c.win && c.kc == 9 * c.cin && c.cin % 32 == 0, "layer shape");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, q = lane >> 4;
  const int gw = blockIdx.x * kConvWaves + wave, group = gw % GROUPS;
  const int ch0 = group * 16 * NT;
  uint4 w[KS][NT];
  float b[4 * NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const uint16_t* row = W + (ch0 + tile_channel<NT>(t, r)) * c.kc + 8 * q;
#pragma unroll
    for (int s = 0; s < KS; ++s) w[s][t] = *reinterpret_cast<const uint4*>(row + 32 * s);
#pragma unroll
    for (int j = 0; j < 4; ++j) b[4 * t + j] = bias[ch0 + 4 * NT * q + 4 * t + j];
  }
  const int stride = gridDim.x * kConvWaves / GROUPS;
  for (int tile = gw / GROUPS; tile * 16 < M; tile += stride) {
    const int m = min(tile * 16 + r, M - 1);  // rows past the end repeat the last one
    const int n = m / (c.hout * c.wout), p = m - n * (c.hout * c.wout);
    const int oy = p / c.wout, ox = p - oy * c.wout;
    const int at = ((n * c.hin + 2 * oy - 1) * c.win + 2 * ox - 1) * c.cin;
    uint4 a[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int tap = 32 * s / c.cin, ky = tap / 3, kx = tap % 3, ci = 32 * s % c.cin + 8 * q;
      const int iy = 2 * oy + ky - 1, ix = 2 * ox + kx - 1;
      const bool in = (ky > 0 || iy >= 0) && (2 * c.hout <= c.hin || iy < c.hin) && (kx > 0 || ix >= 0);
      a[s] = *reinterpret_cast<const uint4*>(X + (in ? at + (ky * c.win + kx) * c.cin + ci : 0));
      if (!in) a[s] = make_uint4(0u, 0u, 0u, 0u);
    }
    v4f acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = mfma32(w[s][t], a[s], acc[t]);
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
      store_bf16<4 * NT>(Yb + o, y);
    }
  }
}

// Input gradient of layer L (1..3), ReLU mask of the layer below and that layer's bias
// sums in one pass: dX[n][iy][ix][ci] = sum over the taps (ky, kx) that reach the
// pixel, in that order, of sum_co dY[n][oy][ox][co] W[co][(ky, kx, ci)]; 0 where the
// forward map Xb is not positive.  A wave takes 16 2x2 pixel blocks (rows 2j, 2j + 1,
// columns 2i, 2i + 1): with stride 2 their nine taps read only the four output pixels
// (j .. j + 1, i .. i + 1), so dY is read four times and every product is needed.
// The weights ([tap][ci][co], so that eight co are one vector) stay in 144 registers.
// Each tap's product is an MFMA chain of its own from zero and the taps are added in
// FP32: the bits of a column-gradient GEMM followed by col2im, without the FP32 column
// matrix (354 MB for layer 2 at batch 256).  bpart: per block and channel the FP32 sum
// of the unrounded gradients.  Batch 256: layers 2 / 3 / 4 in 65 / 34 / 27 us (layer 2:
// 197 MB through memory); the GEMM, col2im, conversion and column sums took 4.3 ms.
template <int L, int NT>
__global__ __launch_bounds__(kConvThreads, 2) void conv_dgrad(const uint16_t* dY, const uint16_t* Wt, const uint16_t* Xb,
                                                              uint16_t* dX, float* bpart, int M) {
  constexpr ConvShape c = kConv[L];
  constexpr int KS = c.cout / 32, GROUPS = c.cin / (16 * NT), CH = 4 * NT;
  static_assert(c.win == 2 * c.wout && (c.hin == 2 * c.hout || c.hin == 2 * c.hout - 1) && kConvWaves % GROUPS == 0,
                "layer shape");
  __shared__ float s_b[kConvWaves][16 * NT];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, q = lane >> 4;
  const int gw = blockIdx.x * kConvWaves + wave, group = gw % GROUPS;
  const int ch0 = group * 16 * NT;
  uint4 w[9][KS][NT];
#pragma unroll
  for (int tap = 0; tap < 9; ++tap)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int s = 0; s < KS; ++s)
        w[tap][s][t] = *reinterpret_cast<const uint4*>(Wt + (tap * c.cin + ch0 + tile_channel<NT>(t, r)) * c.cout + 32 * s + 8 * q);
  float bs[CH];
#pragma unroll
  for (int j = 0; j < CH; ++j) bs[j] = 0.0f;
  const int stride = gridDim.x * kConvWaves / GROUPS;
  for (int tile = gw / GROUPS; tile * 16 < M; tile += stride) {
    const bool live = tile * 16 + r < M;
    const int m = live ? tile * 16 + r : M - 1;
    const int n = m / (c.hout * c.wout), p = m - n * (c.hout * c.wout);
    const int j = p / c.wout, i = p - j * c.wout;
    uint4 a[2][2][KS];  // dY at (j + dj, i + di), 0 outside the map
#pragma unroll
    for (int dj = 0; dj < 2; ++dj)
#pragma unroll
      for (int di = 0; di < 2; ++di) {
        const bool in = (dj == 0 || j + 1 < c.hout) && (di == 0 || i + 1 < c.wout);
        const uint16_t* src = dY + (in ? (m + dj * c.wout + di) * c.cout : 0) + 8 * q;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          a[dj][di][s] = *reinterpret_cast<const uint4*>(src + 32 * s);
          if (!in) a[dj][di][s] = make_uint4(0u, 0u, 0u, 0u);
        }
      }
#pragma unroll
    for (int py = 0; py < 2; ++py)
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
        const int iy = 2 * j + py, ix = 2 * i + px;
        if (live && (c.hin == 2 * c.hout || iy < c.hin)) {
          const int o = ((n * c.hin + iy) * c.win + ix) * c.cin + ch0 + CH * q;
          uint16_t x[CH];
          __builtin_memcpy(x, __builtin_assume_aligned(Xb + o, 2 * CH), 2 * CH);
#pragma unroll
          for (int e = 0; e < CH; ++e) {
            sum[e] = (int16_t)x[e] > 0 ? sum[e] : 0.0f;
            bs[e] = bs[e] + sum[e];
          }
          store_bf16<CH>(dX + o, sum);
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
    bpart[(long)blockIdx.x * c.cin + threadIdx.x] = v;
  }
}

// Sums of partial planes, several at once: out[i] = sum over p < planes of
// part[p * count + i].  A block takes 64 outputs; its sixteen waves each add every
// sixteenth plane (eight loads in flight), and the sixteen sums are added in order.
constexpr int kReduceJobs = 8;
struct ReduceArgs {
  const float* part[kReduceJobs];
  float* out[kReduceJobs];
  int planes[kReduceJobs], count[kReduceJobs], block0[kReduceJobs + 1];
  int jobs;
};

__global__ __launch_bounds__(1024) void reduce_parts(ReduceArgs a) {
  __shared__ float s_v[16][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int k = 0;
  while (k + 1 < a.jobs && (int)blockIdx.x >= a.block0[k + 1]) ++k;
  const int i = ((int)blockIdx.x - a.block0[k]) * 64 + lane, count = a.count[k], planes = a.planes[k];
  const float* src = a.part[k] + min(i, count - 1);
  float sum = 0.0f;
  for (int p = wave; p < planes; p += 128) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = p + 16 * u < planes ? src[(long)(p + 16 * u) * count] : 0.0f;
#pragma unroll
    for (int u = 0; u < 8; ++u) sum = sum + v[u];
  }
  s_v[wave][lane] = sum;
  __syncthreads();
  if (wave == 0 && i < count) {
    for (int u = 1; u < 16; ++u) sum = sum + s_v[u][lane];
    a.out[k][i] = sum;
  }
}

}  // namespace kf
