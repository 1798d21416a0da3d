// kf_prior_head.hpp — the training step's fully connected layers: everything between
// layer 4's activations and their gradients for one sample in one block, the operand
// copies of the weights, and the sums over samples and partial planes that end the step.
#pragma once

#include "kf_prior_conv.hpp"

namespace kf {

constexpr int kFc1Pad = 160;      // FC1 K (134) rounded up to the MFMA step
constexpr int kDoSumPitch = 8;    // row of FP32 output gradients (their sums take four at a time)

// BF16 copies of the weights.  The first holds the blob, layers 2-4 of the convolutions as
// operands (operand_at).  The second (padding zero): per tap of the convolutions an operand
// copy with rows ci and k = co at the blob's offsets, then operand copies of layer 1 with 32
// columns, of FC1 with 160 and of FC1 transposed, and FC2 transposed with rows of 8.
struct WeightCopies {
  long w1, w5, w5t, w6t, total;
  WeightCopies() {
    w1 = (layout().total + 7) / 8 * 8;
    w5 = w1 + kConv[0].cout * 32;
    w5t = w5 + kHidden * kFc1Pad;
    w6t = w5t + kFeat * kHidden;
    total = w6t + kHidden * 8;
  }
};
inline const WeightCopies& weight_copies() {
  static const WeightCopies c;
  return c;
}

struct WeightCopyArgs {
  uint16_t *y, *yt;  // the two copies
  long n, w[6], w1, w5, w5t, w6t;
};

// Parameter i has the value x: its BF16 copies.
__device__ __forceinline__ void copy_weight(const WeightCopyArgs& a, long i, float x) {
  const uint16_t v = bf16_rne(x);
  long at = i;
#pragma unroll
  for (int l = 1; l < kConvs; ++l) {
    const int e = (int)(i - a.w[l]), co = e / kConv[l].kc, k = e - co * kConv[l].kc;
    if (e >= 0 && e < kConv[l].cout * kConv[l].kc) {
      const int tap = k / kConv[l].cin, ci = k - tap * kConv[l].cin;
      at = a.w[l] + operand_at(kConv[l].cout, co, k);
      a.yt[a.w[l] + tap * kConv[l].cin * kConv[l].cout + operand_at(kConv[l].cin, ci, co)] = v;
    }
  }
  a.y[at] = v;
  const int f = (int)(i - a.w[4]), g = (int)(i - a.w[5]), h = (int)(i - a.w[0]);
  if (h >= 0 && h < kConv[0].cout * kConv[0].kc)
    a.yt[a.w1 + operand_at(kConv[0].cout, h / kConv[0].kc, h % kConv[0].kc)] = v;
  if (f >= 0 && f < kHidden * kFc1In) {
    const int row = f / kFc1In, col = f - row * kFc1In;
    a.yt[a.w5 + operand_at(kHidden, row, col)] = v;
    if (col < kFeat) a.yt[a.w5t + operand_at(kFeat, col, row)] = v;
  }
  if (g >= 0 && g < kTwist * kHidden) a.yt[a.w6t + g % kHidden * 8 + g / kHidden] = v;
}

// The forward head of sample n: pooling (the 80 pixels added in order), FC1, FC2 and the
// skip connection, by a block of WAVES wavefronts.  Every product is the MFMA sequence of
// a GEMM over the batch (k steps of 32 from zero); the sample's row is broadcast to the
// 16 rows of the A operand and row 0 of the result is used.  load() issues the weights'
// loads, so that a caller can put them ahead of other latencies.  AGENT: Y4 was written
// by other blocks of the same launch, with agent-scope stores.
template <int WAVES, bool AGENT>
struct HeadForward {
  static constexpr int NT = kHidden / 16 / WAVES;  // FC1 column tiles of a wave
  uint4 w5[NT][kFc1Pad / 32], w6[kHidden / 32];
  float b5[NT], b6;

  __device__ __forceinline__ void load(const uint16_t* W5, const uint16_t* W6, const float* B5, const float* B6) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, q = lane >> 4;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int nn = (wave + WAVES * t) * 16 + r;
#pragma unroll
      for (int s = 0; s < kFc1Pad / 32; ++s) w5[t][s] = *reinterpret_cast<const uint4*>(W5 + operand_at(kHidden, nn, 32 * s + 8 * q));
      b5[t] = B5[nn];
    }
    const int row = min(r, kTwist - 1);  // columns past the six outputs are not used
    if (wave == 0) {                     // FC2 is the first wave's
#pragma unroll
      for (int s = 0; s < kHidden / 32; ++s) w6[s] = *reinterpret_cast<const uint4*>(W6 + row * kHidden + 32 * s + 8 * q);
    }
    b6 = B6[row];
  }

  // xs[kFc1Pad], hs[kHidden] (LDS): FC1's and FC2's inputs.  Returns output r in the
  // lanes q = 0, r < 6 of wave 0; hs is published, the output is not.
  __device__ __forceinline__ float run(const float* Y4, const float* prev, int n, uint16_t* xs, uint16_t* hs) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, q = lane >> 4;
    if (tid < kFc1Pad) {
      float v = 0.0f;
      if (tid < kFeat) {
        const float* y = Y4 + (long)n * kPool * kFeat + tid;
        float e[kPool];  // one round of memory latency
#pragma unroll
        for (int p = 0; p < kPool; ++p) {
          if constexpr (AGENT) e[p] = __hip_atomic_load(const_cast<float*>(y) + p * kFeat, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          else e[p] = y[p * kFeat];
        }
#pragma unroll
        for (int p = 0; p < kPool; ++p) v = v + e[p];
        v = v * (1.0f / (float)kPool);
      } else if (tid < kFc1In) {
        v = prev[n * kTwist + (tid - kFeat)];
      }
      xs[tid] = bf16_rne(v);
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NT; ++t) {  // H = ReLU(X5 W5^T + b5)
      v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int s = 0; s < kFc1Pad / 32; ++s) acc = mfma32(*reinterpret_cast<const uint4*>(&xs[32 * s + 8 * q]), w5[t][s], acc);
      if (q == 0) hs[(wave + WAVES * t) * 16 + r] = bf16_rne(fmaxf(acc[0] + b5[t], 0.0f));
    }
    __syncthreads();
    float o = 0.0f;
    if (wave == 0) {  // O = (H W6^T + b6) + previous twist
      v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int s = 0; s < kHidden / 32; ++s) acc = mfma32(*reinterpret_cast<const uint4*>(&hs[32 * s + 8 * q]), w6[s], acc);
      o = acc[0] + b6;
      o = o + prev[n * kTwist + min(r, kTwist - 1)];
    }
    return o;
  }
};

// The head alone (batched inference): one sample per block.
__global__ __launch_bounds__(kConvThreads) void head_infer(const float* Y4, const float* prev, const uint16_t* W5,
                                                           const uint16_t* W6, const float* B5, const float* B6, float* out) {
  __shared__ __align__(16) uint16_t xs[kFc1Pad], hs[kHidden];
  HeadForward<kConvWaves, false> head;
  head.load(W5, W6, B5, B6);
  const float o = head.run(Y4, prev, blockIdx.x, xs, hs);
  if (threadIdx.x < kTwist) out[blockIdx.x * kTwist + threadIdx.x] = o;
}

struct HeadArgs {
  const float *Y4, *prev, *target, *b5, *b6;
  const uint16_t *w5, *w6, *w5t, *w6t;
  float *O, *dO, *dH;            // [B][6], [B] rows of 8, [B][256]; the last two summed over samples at the end
  uint16_t *X5b, *Hb, *dOb, *dHb;  // the FC weight gradients' operands ([B] rows of 144, 256, 16, 256)
  uint16_t* dY4;
  float* bpart;                  // [B][128]: each sample's sums of dY4 over its pixels
  float inv;                     // 1 / (6 B)
};

// One sample per block: the forward head, the loss gradient, and back to layer 4
// (dY4[p][c] = dX5[c] / 80 where Y4 > 0).  Latency bound (six dependent stages); one
// launch in place of twelve, 60 us of launches at any batch.  12 us at batch 256.  FC2's
// weights are loaded by the wave that uses them, and FC1's transposed ones and the last
// stage's pixels all at once ahead of their use (batch 19: 68.1 -> 67.0 us for the gradients;
// the first alone: inference at batch 1 11.0 -> 10.6).
__global__ __launch_bounds__(kConvThreads) void head_sample(HeadArgs a) {
  __shared__ __align__(16) uint16_t xs[kFc1Pad], hs[kHidden], dhs[kHidden];
  __shared__ __align__(16) uint16_t dos[8];
  __shared__ float dx[kFeat], red[kFeat];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, q = lane >> 4, n = blockIdx.x;
  HeadForward<kConvWaves, false> head;
  head.load(a.w5, a.w6, a.b5, a.b6);
  if (tid < 8) dos[tid] = 0;
  const float o = head.run(a.Y4, a.prev, n, xs, hs);
  // FC1 transposed, in flight while the loss and FC2's gradient are made
  constexpr int kFeatTiles = kFeat / 16 / kConvWaves;
  uint4 w5t[kFeatTiles][kHidden / 32];
#pragma unroll
  for (int t = 0; t < kFeatTiles; ++t)
#pragma unroll
    for (int k = 0; k < kHidden / 32; ++k)
      w5t[t][k] = *reinterpret_cast<const uint4*>(a.w5t + operand_at(kFeat, (wave + kConvWaves * t) * 16 + r, 32 * k + 8 * q));
  if (tid < kX5Pitch) a.X5b[n * kX5Pitch + tid] = xs[tid];
  a.Hb[n * kHidden + tid] = hs[tid];
  static_assert(kHidden == kConvThreads, "one hidden unit a thread");
  if (wave == 0 && q == 0) {  // dLoss/dO
    uint16_t db = 0;
    if (r < kTwist) {
      const float d = o - a.target[n * kTwist + r];
      const float g = 2.0f * d * a.inv;
      a.O[n * kTwist + r] = o;
      a.dO[n * kDoSumPitch + r] = g;
      db = bf16_rne(g);
      dos[r] = db;
    }
    a.dOb[n * kDoPitch + r] = db;
  }
  __syncthreads();
  const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
  const uint4 od = q == 0 ? *reinterpret_cast<const uint4*>(dos) : zero;
  for (int nt = wave; nt < kHidden / 16; nt += kConvWaves) {  // dH = dO W6 where H > 0
    const int nn = nt * 16 + r;
    v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
    acc = mfma32(od, q == 0 ? *reinterpret_cast<const uint4*>(a.w6t + nn * 8) : zero, acc);
    if (q == 0) {
      const float v = (int16_t)hs[nn] > 0 ? acc[0] : 0.0f;
      dhs[nn] = bf16_rne(v);
      a.dH[n * kHidden + nn] = v;
      a.dHb[n * kHidden + nn] = dhs[nn];
    }
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < kFeatTiles; ++t) {  // dX5 = dH W5 (the pooled features)
    v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < kHidden / 32; ++k) acc = mfma32(*reinterpret_cast<const uint4*>(&dhs[32 * k + 8 * q]), w5t[t][k], acc);
    if (q == 0) dx[(wave + kConvWaves * t) * 16 + r] = acc[0];
  }
  __syncthreads();
  const int c = tid & (kFeat - 1), half = tid / kFeat;
  const float g = dx[c] * (1.0f / (float)kPool);
  const uint16_t gb = bf16_rne(g);
  float s = 0.0f;
  const float* y = a.Y4 + ((long)n * kPool + half) * kFeat + c;
  float e[kPool / 2];  // one round of memory latency
#pragma unroll
  for (int p = 0; p < kPool / 2; ++p) e[p] = y[2 * p * kFeat];
  uint16_t* dy = a.dY4 + ((long)n * kPool + half) * kFeat + c;
#pragma unroll
  for (int p = 0; p < kPool / 2; ++p) {
    const bool on = e[p] > 0.0f;
    dy[2 * p * kFeat] = on ? gb : (uint16_t)0;
    s = s + (on ? g : 0.0f);
  }
  if (half == 1) red[c] = s;
  __syncthreads();
  if (half == 0) a.bpart[(long)n * kFeat + c] = s + red[c];
}

// The end of the backward pass: sums of partial planes, several at once, out[i] = sum
// over p < planes of part[p * pitch + i].  A lane takes four outputs (16-byte loads, 256
// outputs a block); the block's sixteen waves each add every sixteenth plane (eight
// loads in flight) in FP64.  Bound by memory: 58 MB of planes at batch 256, 13 us
// (one output a lane took 28 where this took 17).
constexpr int kReduceJobs = 10, kReduceThreads = 1024, kReduceWaves = kReduceThreads / kWave, kReduceOut = 4 * kWave;
struct ReduceArgs {
  const float* part[kReduceJobs];
  float* out[kReduceJobs];
  int planes[kReduceJobs], pitch[kReduceJobs], count[kReduceJobs], block0[kReduceJobs + 1];  // pitch: a multiple of 4
  int jobs;
};

__global__ __launch_bounds__(kReduceThreads, 8) void reduce_parts(ReduceArgs a) {
  __shared__ double s_v[kReduceWaves][kReduceOut];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int k = 0;
  while (k + 1 < a.jobs && (int)blockIdx.x >= a.block0[k + 1]) ++k;
  const int i0 = ((int)blockIdx.x - a.block0[k]) * kReduceOut, pitch = a.pitch[k], planes = a.planes[k];
  const float* src = a.part[k] + min(i0 + 4 * lane, pitch - 4);  // lanes past the end repeat the last outputs
  double sum[4] = {0.0, 0.0, 0.0, 0.0};
  for (int p = wave; p < planes; p += 8 * kReduceWaves) {
    float4 v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int at = p + kReduceWaves * u;
      v[u] = *reinterpret_cast<const float4*>(src + (long)min(at, planes - 1) * pitch);
      if (at >= planes) v[u] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      sum[0] = sum[0] + (double)v[u].x;
      sum[1] = sum[1] + (double)v[u].y;
      sum[2] = sum[2] + (double)v[u].z;
      sum[3] = sum[3] + (double)v[u].w;
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) s_v[wave][64 * j + lane] = sum[j];  // output 4 lane + j
  __syncthreads();
  const int i = i0 + 4 * lane + wave;
  if (wave < 4 && i < a.count[k]) {
    double t = 0.0;
#pragma unroll
    for (int u = 0; u < kReduceWaves; ++u) t = t + s_v[u][64 * wave + lane];
    a.out[k][i] = (float)t;
  }
}

}  // namespace kf
