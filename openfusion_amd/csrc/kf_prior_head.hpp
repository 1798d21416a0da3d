// kf_prior_head.hpp — the training step's fully connected layers: everything between
// layer 4's activations and their gradients for one sample in one block, the operand
// copies of the weights, and the sums over samples and partial planes that end the step.
#pragma once

#include "kf_prior_conv.hpp"

namespace kf {

constexpr int kFc1Pad = 160;      // FC1 K (134) rounded up to the MFMA step
constexpr int kDoSumPitch = 8;    // row of FP32 output gradients (their sums take four at a time)

// Second BF16 copies of weights, laid out as operands (padding zero): the convolutions'
// [tap][ci][co] at the blob's offsets, then FC1 with rows of 160, FC1 transposed
// ([feature][hidden]) and FC2 transposed with rows of 8.
struct WeightCopies {
  long w5, w5t, w6t, total;
  WeightCopies() {
    w5 = (layout().total + 7) / 8 * 8;
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
  uint16_t *y, *yt;  // the blob as BF16; the operand copies
  long n, w[6], w5, w5t, w6t;
};

// Parameter i has the value x: its BF16 copies.
__device__ __forceinline__ void copy_weight(const WeightCopyArgs& a, long i, float x) {
  const uint16_t v = bf16_rne(x);
  a.y[i] = v;
#pragma unroll
  for (int l = 1; l < kConvs; ++l) {
    const int e = (int)(i - a.w[l]);
    if (e >= 0 && e < kConv[l].cout * kConv[l].kc) a.yt[a.w[l] + (e % kConv[l].kc) * kConv[l].cout + e / kConv[l].kc] = v;
  }
  const int f = (int)(i - a.w[4]), g = (int)(i - a.w[5]);
  if (f >= 0 && f < kHidden * kFc1In) {
    const int row = f / kFc1In, col = f - row * kFc1In;
    a.yt[a.w5 + row * kFc1Pad + col] = v;
    if (col < kFeat) a.yt[a.w5t + col * kHidden + row] = v;
  }
  if (g >= 0 && g < kTwist * kHidden) a.yt[a.w6t + g % kHidden * 8 + g / kHidden] = v;
}

// Mean of layer 4 over its pixels for feature c of sample n (added in pixel order).
__device__ __forceinline__ float pooled_feature(const float* Y4, int n, int c) {
  constexpr int kLoads = 40;  // two rounds of memory latency
  static_assert(kPool % kLoads == 0, "pooling batches");
  const float* y = Y4 + (long)n * kPool * kFeat + c;
  float s = 0.0f;
  for (int p = 0; p < kPool; p += kLoads) {
    float v[kLoads];
#pragma unroll
    for (int u = 0; u < kLoads; ++u) v[u] = y[(p + u) * kFeat];
#pragma unroll
    for (int u = 0; u < kLoads; ++u) s = s + v[u];
  }
  return s * (1.0f / (float)kPool);
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

// One sample per block: pooling, FC1, FC2 and the skip connection, the loss gradient,
// and back to layer 4 (dY4[p][c] = dX5[c] / 80 where Y4 > 0).  Every product is the
// MFMA sequence of a GEMM over the batch (k steps of 32 from zero); the sample's row is
// broadcast to the 16 rows of the A operand and row 0 of the result is used.  Latency
// bound (six dependent stages); one launch in place of twelve, 60 us of launches at any
// batch.  18 us at batch 256.
__global__ __launch_bounds__(kConvThreads) void head_sample(HeadArgs a) {
  __shared__ __align__(16) uint16_t xs[kFc1Pad], hs[kHidden], dhs[kHidden];
  __shared__ __align__(16) uint16_t dos[8];
  __shared__ float dx[kFeat], red[kFeat];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, q = lane >> 4, n = blockIdx.x;
  if (tid < kFc1Pad) {
    float v = 0.0f;
    if (tid < kFeat) v = pooled_feature(a.Y4, n, tid);
    else if (tid < kFc1In) v = a.prev[n * kTwist + (tid - kFeat)];
    xs[tid] = bf16_rne(v);
    if (tid < kX5Pitch) a.X5b[n * kX5Pitch + tid] = xs[tid];
  }
  if (tid < 8) dos[tid] = 0;
  __syncthreads();
  for (int nt = wave; nt < kHidden / 16; nt += kConvWaves) {  // H = ReLU(X5 W5^T + b5)
    const int nn = nt * 16 + r;
    v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < kFc1Pad; k += 32)
      acc = mfma32(*reinterpret_cast<const uint4*>(&xs[k + 8 * q]),
                   *reinterpret_cast<const uint4*>(a.w5 + nn * kFc1Pad + k + 8 * q), acc);
    if (q == 0) {
      hs[nn] = bf16_rne(fmaxf(acc[0] + a.b5[nn], 0.0f));
      a.Hb[n * kHidden + nn] = hs[nn];
    }
  }
  __syncthreads();
  if (wave == 0) {  // O = (H W6^T + b6) + previous twist, and dLoss/dO
    v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
    const int row = min(r, kTwist - 1);  // columns past the six outputs are not used
#pragma unroll
    for (int k = 0; k < kHidden; k += 32)
      acc = mfma32(*reinterpret_cast<const uint4*>(&hs[k + 8 * q]),
                   *reinterpret_cast<const uint4*>(a.w6 + row * kHidden + k + 8 * q), acc);
    if (q == 0) {
      uint16_t db = 0;
      if (r < kTwist) {
        float v = acc[0] + a.b6[r];
        v = v + a.prev[n * kTwist + r];
        const float d = v - a.target[n * kTwist + r];
        const float g = 2.0f * d * a.inv;
        a.O[n * kTwist + r] = v;
        a.dO[n * kDoSumPitch + r] = g;
        db = bf16_rne(g);
        dos[r] = db;
      }
      a.dOb[n * kDoPitch + r] = db;
    }
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
  for (int nt = wave; nt < kFeat / 16; nt += kConvWaves) {  // dX5 = dH W5 (the pooled features)
    const int nn = nt * 16 + r;
    v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < kHidden; k += 32)
      acc = mfma32(*reinterpret_cast<const uint4*>(&dhs[k + 8 * q]),
                   *reinterpret_cast<const uint4*>(a.w5t + nn * kHidden + k + 8 * q), acc);
    if (q == 0) dx[nn] = acc[0];
  }
  __syncthreads();
  const int c = tid & (kFeat - 1), half = tid / kFeat;
  const float g = dx[c] * (1.0f / (float)kPool);
  const uint16_t gb = bf16_rne(g);
  float s = 0.0f;
#pragma unroll 20
  for (int p = half; p < kPool; p += 2) {
    const long i = ((long)n * kPool + p) * kFeat + c;
    const bool on = a.Y4[i] > 0.0f;
    a.dY4[i] = on ? gb : (uint16_t)0;
    s = s + (on ? g : 0.0f);
  }
  if (half == 1) red[c] = s;
  __syncthreads();
  if (half == 0) a.bpart[(long)n * kFeat + c] = s + red[c];
}

// The end of the backward pass: sums of partial planes, several at once, out[i] = sum
// over p < planes of part[p * pitch + i].  A lane takes four outputs (16-byte loads, 256
// outputs a block); the block's sixteen waves each add every sixteenth plane (eight
// loads in flight) in FP64.  Bound by memory: 58 MB of planes at batch 256, 17 us
// (28 us with one output a lane).
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
