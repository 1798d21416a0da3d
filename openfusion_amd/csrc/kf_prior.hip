// kf_prior.hip — the learned pose prior: CNN inference and training on gfx950.
//
// No counterpart in the reference (its ICP starts from the previous pose,
// Source/src/ICP.cpp:94).  Network: four 3x3 stride-2 pad-1 convolutions
// (2->32->64->64->128, ReLU) on two 160x120 depth maps, global average pooling,
// concatenation with the previous frame's twist, FC 134->256 (ReLU), FC 256->6,
// plus the previous twist (skip connection: the layers predict the change of motion).
//
// Layout: activations NHWC (pixel-major, channel fastest), layers 1-3 as BF16 (the
// next layer's operand), layer 4 FP32; products are BF16 (round to nearest even) with
// FP32 accumulation.  Training's convolutions, their input and weight gradients read
// the maps directly (kf_prior_conv.hpp); its fully connected layers run both ways in one
// block per sample (kf_prior_head.hpp).
#include "kf_prior_head.hpp"

#include <math.h>
#include <string.h>

#include <algorithm>
#include <vector>

namespace kf {
namespace {

// ---------------------------------------------------------------------------
// Fused inference (kf_prior_forward at small batches): one block per (layer-4 pixel,
// sample) carries the pixel's receptive field through the four convolutions in
// LDS — a 15x15 window of layer 1, 7x7 of layer 2, 3x3 of layer 3, then the pixel
// (window positions outside a layer's map hold zeros: that layer's padding) — and
// computes every output with the MFMA sequence training runs for it (k steps of
// 32 from 0 on the same BF16 operands, the same epilogue), so every activation
// equals the layer-by-layer forward's bit for bit.  Neighbouring blocks recompute
// the overlap of their windows (~2.7x the 42 M MACs of one sample) in exchange for
// one launch, with nothing between the layers but LDS.  The last
// block of a sample to finish (a device counter, cleared again by that block)
// runs the forward head.
//
// Bound by latency: at batch 1 there are 80 blocks and every stage waits for the one
// before.  So the weights are the A operand, held in registers and loaded a layer ahead
// of their use; eight waves share each layer's tiles; window pixels are padded by 16
// bytes in LDS (without, the 16 pixels of an operand read lie on the same banks); the
// layer-4 pixels go to the last block by agent-scope stores and loads (no L2 write-back
// and invalidation, kf_icp.hip), all of them in flight together.  Batch 1: 10.6 us (17.6
// with the weights' rows on end; 23.7 with four waves, weights loaded where they are used,
// scalar FC1 weight loads and fences around the hand-over).
constexpr int kFuseThreads = 512, kFuseWaves = kFuseThreads / kWave;
constexpr int kWin1 = 15, kWin2 = 7, kWin3 = 3;  // window sides of layers 1-3 around one layer-4 pixel
constexpr int kRows1 = kWin1 * kWin1;            // 225 layer-1 positions
constexpr int kPatch = 2 * kWin1 + 1;            // 31: input window side
constexpr int kPix1 = 32 + 8, kPix2 = 64 + 8, kPix3 = 64;  // elements per window pixel in LDS

struct FuseArgs {
  const float* frames;
  const int32_t* pairs;
  const float* prev;
  const uint16_t* wbf;   // BF16 weights
  const uint16_t *w1, *w5;  // operand copies of layer 1 and FC1 (WeightCopies)
  const float* params;   // FP32 biases
  long w[6], b[6];       // parameter offsets
  float* Y4;             // [B][80][128] layer-4 activations
  float* out;            // [B][6]
  unsigned* count;       // [B] finished blocks of each sample (zero between calls)
};

// NT tiles of one convolution layer (L 1..3) as a wave computes them: channels ch0 .. of
// 16 window positions.  Output window side WOUT; input window pixels of PIN elements.
template <int L, int NT, int WOUT, int PIN>
struct FuseConv {
  static constexpr ConvShape c = kConv[L];
  static constexpr int KS = c.kc / 32, CH = 4 * NT;
  uint4 w[KS][NT];
  float b[CH];

  __device__ __forceinline__ void load(const uint16_t* W, const float* bias, int ch0) {
    const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
      for (int s = 0; s < KS; ++s)
        w[s][t] = *reinterpret_cast<const uint4*>(W + operand_at(c.cout, ch0 + tile_channel<NT>(t, r), 32 * s + 8 * q));
#pragma unroll
      for (int j = 0; j < 4; ++j) b[4 * t + j] = bias[ch0 + CH * q + 4 * t + j];
    }
  }

  // Channels ch0 + CH q .. of position p (in the window); y: ReLU(conv + bias).
  __device__ __forceinline__ void run(const uint16_t* in, int p, float* y) const {
    const int q = (threadIdx.x & 63) >> 4;
    const int wy = p / WOUT, wx = p - wy * WOUT;
    const uint16_t* at = in + (2 * wy * (2 * WOUT + 1) + 2 * wx) * PIN + 8 * q;
    v4f acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int tap = 32 * s / c.cin, ci = 32 * s % c.cin;
      const uint4 a = *reinterpret_cast<const uint4*>(at + (tap / 3 * (2 * WOUT + 1) + tap % 3) * PIN + ci);
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t] = mfma32(w[s][t], a, acc[t]);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) y[4 * t + j] = fmaxf(acc[t][j] + b[4 * t + j], 0.0f);
  }

  // The same, stored as BF16 into the output window (POUT elements per pixel) with origin
  // (y0, x0) in the layer's map, zero outside it.
  template <int POUT>
  __device__ __forceinline__ void run_store(const uint16_t* in, int tile, uint16_t* out, int ch0, int y0, int x0) const {
    const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const int p = tile * 16 + r;
    float y[CH];
    run(in, min(p, WOUT * WOUT - 1), y);
    if (p >= WOUT * WOUT) return;
    const int gy = y0 + p / WOUT, gx = x0 + p % WOUT;
    if (!(gy >= 0 && gy < c.hout && gx >= 0 && gx < c.wout)) {
#pragma unroll
      for (int j = 0; j < CH; ++j) y[j] = 0.0f;
    }
    store_bf16<CH>(out + p * POUT + ch0 + CH * q, y);
  }
};

__global__ __launch_bounds__(kFuseThreads) void prior_infer_fused(FuseArgs f) {
  __shared__ uint32_t patch[kPatch][kPatch + 1];  // input window, BF16 pairs (previous, current)
  __shared__ __align__(16) uint16_t act1[kRows1 * kPix1];  // layer windows, NHWC
  __shared__ __align__(16) uint16_t act2[kWin2 * kWin2 * kPix2];
  __shared__ __align__(16) uint16_t act3[kWin3 * kWin3 * kPix3];
  __shared__ __align__(16) uint16_t xs[kFc1Pad], hs[kHidden];
  __shared__ int s_last;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, q = lane >> 4;
  const int n = blockIdx.y, pix = blockIdx.x;
  const int y4 = pix / kConv[3].wout, x4 = pix - y4 * kConv[3].wout;
  const float* f0 = f.frames + (long)f.pairs[2 * n] * (kH0 * kW0);
  const float* f1 = f.frames + (long)f.pairs[2 * n + 1] * (kH0 * kW0);

  // the 31x31 input window (zero outside the frame): the loads first, the weights of
  // layers 1 and 2 behind them
  constexpr int E = kPatch * kPatch, PER = (E + kFuseThreads - 1) / kFuseThreads;
  float v[PER][2];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int e = tid + kFuseThreads * u, py = e / kPatch, px = e - py * kPatch;
    const int iy = 16 * y4 - 15 + py, ix = 16 * x4 - 15 + px;
    const bool in = e < E && iy >= 0 && iy < kH0 && ix >= 0 && ix < kW0;
    const int o = in ? iy * kW0 + ix : 0;
    v[u][0] = in ? f0[o] : 0.0f;
    v[u][1] = in ? f1[o] : 0.0f;
  }
  uint4 w1[2];
  float b1[8];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    w1[t] = conv1_weights(f.w1, t, r, q);
#pragma unroll
    for (int j = 0; j < 4; ++j) b1[4 * t + j] = f.params[f.b[0] + 8 * q + 4 * t + j];
  }
  FuseConv<1, 2, kWin2, kPix1> c2;  // wave: channels 32 (wave / 4) .., position tile wave % 4
  const int ch2 = wave / 4 * 32;
  c2.load(f.wbf + f.w[1], f.params + f.b[1], ch2);
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int e = tid + kFuseThreads * u;
    if (e < E) patch[e / kPatch][e % kPatch] = pack_bf16(v[u][0], v[u][1]);
  }
  __syncthreads();
  FuseConv<2, 1, kWin3, kPix2> c3;  // waves 0..3: channels 16 wave ..
  const int ch3 = wave % 4 * 16;
  c3.load(f.wbf + f.w[2], f.params + f.b[2], ch3);
  {  // layer 1: one K step, the lane's four taps straight from the patch (tap 8 alone at q = 2)
    int off[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int tap = min(4 * q + e, 8);
      off[e] = tap / 3 * (kPatch + 1) + tap % 3;
    }
    for (int tile = wave; tile < (kRows1 + 15) / 16; tile += kFuseWaves) {
      const int p = tile * 16 + r, pc = min(p, kRows1 - 1), wy = pc / kWin1, wx = pc - wy * kWin1;
      const uint32_t* at = &patch[0][0] + 2 * wy * (kPatch + 1) + 2 * wx;
      uint32_t a[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        a[e] = at[off[e]];
        if (4 * q + e > 8) a[e] = 0u;
      }
      const int gy = 8 * y4 - 7 + wy, gx = 8 * x4 - 7 + wx;
      const bool in_map = gy >= 0 && gy < kConv[0].hout && gx >= 0 && gx < kConv[0].wout;
      float y[8];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
        acc = mfma32(w1[t], make_uint4(a[0], a[1], a[2], a[3]), acc);
#pragma unroll
        for (int j = 0; j < 4; ++j) y[4 * t + j] = in_map ? fmaxf(acc[j] + b1[4 * t + j], 0.0f) : 0.0f;
      }
      if (p < kRows1) store_bf16<8>(act1 + p * kPix1 + 8 * q, y);
    }
  }
  __syncthreads();
  c2.run_store<kPix2>(act1, wave % 4, act2, ch2, 4 * y4 - 3, 4 * x4 - 3);
  FuseConv<3, 1, 1, kPix3> c4;  // wave: channels 16 wave ..
  const int ch4 = wave * 16;
  c4.load(f.wbf + f.w[3], f.params + f.b[3], ch4);
  __syncthreads();
  if (wave < 4) c3.run_store<kPix3>(act2, 0, act3, ch3, 2 * y4 - 1, 2 * x4 - 1);
  __syncthreads();
  {
    float y[4];
    c4.run(act3, 0, y);
    float* o = f.Y4 + ((long)n * kPool + pix) * kFeat + ch4 + 4 * q;
    if (r == 0) {
#pragma unroll
      for (int j = 0; j < 4; ++j) __hip_atomic_store(o + j, y[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }

  // the last block of the sample: every block's stores have completed (s_waitcnt 0
  // counts them) before its arrival, and the loads below are agent-scope too
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (tid == 0)
    s_last = __hip_atomic_fetch_add(&f.count[n], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(kPool - 1);
  __syncthreads();
  if (!s_last) return;  // uniform
  HeadForward<kFuseWaves, true> head;
  head.load(f.w5, f.wbf + f.w[5], f.params + f.b[4], f.params + f.b[5]);
  const float o = head.run(f.Y4, f.prev, n, xs, hs);
  if (tid < kTwist) f.out[n * kTwist + tid] = o;
  if (tid == 0) f.count[n] = 0u;  // ready for the next call
}

__global__ void copy_weights(WeightCopyArgs a, const float* p) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < a.n) copy_weight(a, i, p[i]);
}

// One Adam step; the new parameters' BF16 copies are made with it.
__global__ void adam(WeightCopyArgs w, float* p, const float* g, float* m, float* v, long n, float lr, float b1,
                     float b2, float eps, float c1, float c2) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  p[i] = pi;
  copy_weight(w, i, pi);
}

inline unsigned blocks_for(long n, int t = 256) { return (unsigned)((n + t - 1) / t); }

}  // namespace
}  // namespace kf

struct kf_prior {
  int max_batch = 0;
  long nparams = 0;
  float* params = nullptr;   // FP32 master
  uint16_t* wbf = nullptr;   // BF16 copy
  uint16_t* wt = nullptr;    // operand copies (WeightCopies)
  float* grad = nullptr;
  float* adam_m = nullptr;
  float* adam_v = nullptr;
  long step = 0;
  // activations (NHWC), sized for max_batch
  uint16_t* Yb[kf::kConvs - 1] = {};  // layers 1-3, BF16 NHWC
  uint8_t* signs[kf::kConvs - 1] = {};  // bit i of byte b: value 8 b + i of Yb is positive
  float* Y4 = nullptr;                // layer 4, FP32
  uint16_t* X5b = nullptr;
  uint16_t* Hb = nullptr;
  float* O = nullptr;
  float* dO = nullptr;
  uint16_t* dOb = nullptr;
  float* dH = nullptr;
  uint16_t* dHb = nullptr;
  uint16_t* dYb[kf::kConvs] = {};       // gradients of the layers' outputs, BF16 NHWC
  float* bpart[kf::kConvs] = {};        // partial bias sums per block (layer 4: per sample)
  float* wpart[kf::kConvs] = {};        // partial weight gradients per split
  unsigned* fuse_count = nullptr;  // [max_batch] finished blocks per sample of the fused inference
};

namespace kf {
namespace {

// BF16 copies of the weights; every call that changes the FP32 parameters refreshes
// them, so inference (forward) never converts.
WeightCopyArgs copy_args(kf_prior* P) {
  WeightCopyArgs a;
  a.y = P->wbf;
  a.yt = P->wt;
  a.n = P->nparams;
  for (int q = 0; q < 6; ++q) a.w[q] = layout().w[q];
  a.w1 = weight_copies().w1;
  a.w5 = weight_copies().w5;
  a.w5t = weight_copies().w5t;
  a.w6t = weight_copies().w6t;
  return a;
}

kf_status sync_weights(kf_prior* P, hipStream_t s) {
  hipLaunchKernelGGL(copy_weights, dim3(blocks_for(P->nparams)), dim3(256), 0, s, copy_args(P), (const float*)P->params);
  return check_launch("copy_weights");
}

constexpr int kConvBlocks = 512;

// One convolution of the training forward: two blocks of four waves a CU hold the
// weights; a small batch gets one wave per 16-pixel tile and channel group.
template <int L, int NT, bool F32>
kf_status launch_conv(kf_prior* P, const uint16_t* X, uint16_t* Yb, float* Y, uint8_t* signs, int B, hipStream_t s) {
  constexpr ConvShape c = kConv[L];
  constexpr int GROUPS = c.cout / (16 * NT);
  const ParamLayout& lay = layout();
  const int M = B * c.hout * c.wout;
  const int blocks = std::min(div_up(div_up(M, 16) * GROUPS, kConvWaves), kConvBlocks);
  hipLaunchKernelGGL((conv_forward<L, NT, F32>), dim3(blocks), dim3(kConvThreads), 0, s, X, P->wbf + lay.w[L],
                     (const float*)P->params + lay.b[L], Yb, Y, signs, M);
  return check_launch("conv_forward");
}

// Training forward of the convolutions: the activations stay for the backward pass, and
// (train) the signs of layers 1-3.
kf_status forward(kf_prior* P, const float* frames, const int32_t* pairs, int B, bool train, hipStream_t s) {
  const ParamLayout& L = layout();
  uint8_t* none[kConvs - 1] = {};
  uint8_t* const* signs = train ? P->signs : none;
  hipLaunchKernelGGL(conv1_forward, dim3(kConv[0].hout / kL1Rows, B), dim3(kConvThreads), 0, s, frames, pairs,
                     (const uint16_t*)P->wt + weight_copies().w1, (const float*)P->params + L.b[0], P->Yb[0], signs[0]);
  KF_TRY(check_launch("conv1_forward"));
  KF_TRY((launch_conv<1, 4, false>(P, P->Yb[0], P->Yb[1], nullptr, signs[1], B, s)));
  KF_TRY((launch_conv<2, 2, false>(P, P->Yb[1], P->Yb[2], nullptr, signs[2], B, s)));
  return launch_conv<3, 2, true>(P, P->Yb[2], nullptr, P->Y4, nullptr, B, s);
}

// Inference, with the training forward's outputs either way.  The fused kernel's blocks
// (80 a sample, one fits a CU) are all resident up to three samples on 256 CUs; from the
// fourth on they take a second round, and from the sixth on that and the recomputed window
// overlaps cost more than the layered forward's five launches.  Fused / layered at batch 1:
// 10.7 / 19.5 us, 3: 12.8 / 19.9, 4: 18.4 / 20.1, 5: 19.2 / 20.4, 6: 21.1 / 20.7, 8: 26.0 / 20.9.
constexpr int kLayeredBatch = 6;
kf_status infer(kf_prior* P, const float* frames, const int32_t* pairs, const float* prev, int B, float* out,
                hipStream_t s) {
  const ParamLayout& L = layout();
  if (B >= kLayeredBatch) {
    KF_TRY(forward(P, frames, pairs, B, false, s));
    hipLaunchKernelGGL(head_infer, dim3(B), dim3(kConvThreads), 0, s, (const float*)P->Y4, prev,
                       (const uint16_t*)P->wt + weight_copies().w5, (const uint16_t*)P->wbf + L.w[5],
                       (const float*)P->params + L.b[4], (const float*)P->params + L.b[5], out);
    return check_launch("head_infer");
  }
  FuseArgs f;
  f.frames = frames;
  f.pairs = pairs;
  f.prev = prev;
  f.wbf = P->wbf;
  f.w1 = P->wt + weight_copies().w1;
  f.w5 = P->wt + weight_copies().w5;
  f.params = P->params;
  for (int q = 0; q < 6; ++q) {
    f.w[q] = L.w[q];
    f.b[q] = L.b[q];
  }
  f.Y4 = P->Y4;
  f.out = out;
  f.count = P->fuse_count;
  hipLaunchKernelGGL(prior_infer_fused, dim3(kPool, B), dim3(kFuseThreads), 0, s, f);
  return check_launch("prior_infer_fused");
}

// Backward pass of layer L: the weight gradient as *splits partial planes, one block a CU
// and at least kWgradMinSteps steps of 32 pixels each (a shorter split would mostly
// write its plane), and dYb[L] -> dYb[L - 1] with *planes partial sums of layer L - 1's
// bias gradient, one block a CU beside the first: two blocks fit a CU, so all are
// resident at once (512 blocks of input gradient ran a second round: 179 us against 159
// for the three layers at batch 256).  fc (L = 1): carried along.
// Layer 2's input gradient, which also makes layer 1's weight gradient, takes longer than
// its weight gradient: from eight tiles a wave on it gets 320 of the 512 blocks (batch 256:
// 58.9 us against 66.8; with few tiles a block mostly loads its weights, and 256 are the
// better: batch 19 11.6 us against 12.6).
constexpr int kWgradBlocks = 256, kWgradMinSteps = 4, kDgradBlocks = 256, kDgradMore = 320;
template <int L>
kf_status launch_backward(kf_prior* P, int B, int* splits, int* planes, hipStream_t s, const FcGradArgs& fc = FcGradArgs{},
                          const Conv1Grad& first = Conv1Grad{}) {
  constexpr int GROUPS = WgradShape<L>::GROUPS;
  const int M = B * kConv[L].hout * kConv[L].wout, steps = div_up(M, kWgradStep);
  const int units = div_up(div_up(M, 16) * DgradShape<L>::GROUPS, kConvWaves);  // blocks at one tile a wave
  const int most = L == 1 && units >= 8 * kDgradMore ? kDgradMore : kDgradBlocks;
  const int want = std::min(std::max(steps / kWgradMinSteps, 1), (kWgradBlocks + kDgradBlocks - most) / GROUPS);
  ConvBackArgs a;
  a.dY = P->dYb[L];
  a.X = P->Yb[L - 1];
  a.signs = P->signs[L - 1];
  a.Wt = P->wt + layout().w[L];
  a.dX = P->dYb[L - 1];
  a.wpart = P->wpart[L];
  a.bpart = P->bpart[L - 1];
  a.M = M;
  a.steps_per_split = div_up(steps, want);
  *splits = div_up(steps, a.steps_per_split);
  // eight splits a round (blocks of one split on one XCD): the count is rounded up, and
  // the splits past the last write zero planes that nothing reads
  a.wblocks = div_up(*splits, 8) * 8 * GROUPS;
  a.dblocks = *planes = std::min(units, most);
  a.fc = fc;
  a.first = first;
  hipLaunchKernelGGL(conv_backward<L>, dim3(a.wblocks + a.dblocks + (L == 1 ? kFcBlocks : 0)), dim3(kConvThreads), 0, s, a);
  return check_launch("conv_backward");
}

// The fully connected layers both ways, then the convolutions' backward; the gradient
// of every parameter goes to G.
kf_status backward(kf_prior* P, const float* frames, const int32_t* pairs, const float* prev, const float* target, int B,
                   float* G, float* loss, hipStream_t s) {
  const ParamLayout& L = layout();
  const WeightCopies& W = weight_copies();
  HeadArgs h;
  h.Y4 = P->Y4;
  h.prev = prev;
  h.target = target;
  h.b5 = P->params + L.b[4];
  h.b6 = P->params + L.b[5];
  h.w5 = P->wt + W.w5;
  h.w6 = P->wbf + L.w[5];
  h.w5t = P->wt + W.w5t;
  h.w6t = P->wt + W.w6t;
  h.O = P->O;
  h.dO = P->dO;
  h.dH = P->dH;
  h.X5b = P->X5b;
  h.Hb = P->Hb;
  h.dOb = P->dOb;
  h.dHb = P->dHb;
  h.dY4 = P->dYb[3];
  h.bpart = P->bpart[3];
  h.inv = 1.0f / (float)(B * kTwist);
  hipLaunchKernelGGL(head_sample, dim3(B), dim3(kConvThreads), 0, s, h);
  KF_TRY(check_launch("head_sample"));
  int planes[kConvs] = {0, 0, 0, B}, splits[kConvs];
  KF_TRY(launch_backward<3>(P, B, &splits[3], &planes[2], s));
  KF_TRY(launch_backward<2>(P, B, &splits[2], &planes[1], s));
  FcGradArgs fc;
  fc.X5b = P->X5b;
  fc.Hb = P->Hb;
  fc.dOb = P->dOb;
  fc.dHb = P->dHb;
  fc.O = P->O;
  fc.target = target;
  fc.dW5 = G + L.w[4];
  fc.dW6 = G + L.w[5];
  fc.loss = loss;
  fc.batch = B;
  KF_TRY(launch_backward<1>(P, B, &splits[1], &planes[0], s, fc, Conv1Grad{frames, pairs, P->wpart[0]}));
  splits[0] = planes[0];
  ReduceArgs f;
  f.jobs = 0;
  f.block0[0] = 0;
  auto add = [&](const float* part, int n, int pitch, int count, float* out) {
    const int k = f.jobs++;
    f.part[k] = part;
    f.planes[k] = n;
    f.pitch[k] = pitch;
    f.count[k] = count;
    f.out[k] = out;
    f.block0[k + 1] = f.block0[k] + div_up(count, kReduceOut);
  };
  for (int l = 0; l < kConvs; ++l) {
    const int nw = kConv[l].cout * kConv[l].kc;
    add(P->wpart[l], splits[l], nw, nw, G + L.w[l]);
    add(P->bpart[l], planes[l], kConv[l].cout, kConv[l].cout, G + L.b[l]);
  }
  add(P->dH, B, kHidden, kHidden, G + L.b[4]);
  add(P->dO, B, kDoSumPitch, kTwist, G + L.b[5]);
  hipLaunchKernelGGL(reduce_parts, dim3(f.block0[f.jobs]), dim3(kReduceThreads), 0, s, f);
  return check_launch("reduce_parts");
}

kf_status check_batch(const kf_prior* P, const float* frames, const int32_t* pairs, const float* prev, int B) {
  KF_CHECK_ARG(P && frames && pairs && prev, "NULL argument");
  KF_CHECK_ARG(B >= 1 && B <= P->max_batch, "batch must be 1..max_batch");
  return KF_OK;
}

}  // namespace
}  // namespace kf

using namespace kf;

extern "C" int64_t kf_prior_param_count(void) { return layout().total; }

extern "C" kf_status kf_prior_destroy(kf_prior* P) {
  if (!P) return KF_OK;
  void* ptrs[] = {P->params, P->wbf, P->grad, P->adam_m, P->adam_v, P->Y4, P->X5b, P->Hb, P->O, P->dO,
                  P->dOb, P->dH, P->dHb, P->wt, P->fuse_count};
  for (void* q : ptrs) (void)hipFree(q);
  for (int l = 0; l < kConvs; ++l) {
    if (l + 1 < kConvs) {
      (void)hipFree(P->Yb[l]);
      (void)hipFree(P->signs[l]);
    }
    (void)hipFree(P->wpart[l]);
    (void)hipFree(P->dYb[l]);
    (void)hipFree(P->bpart[l]);
  }
  delete P;
  return KF_OK;
}

extern "C" kf_status kf_prior_create(int32_t max_batch, kf_prior** out) {
  KF_CHECK_ARG(out != nullptr, "out is NULL");
  KF_CHECK_ARG(max_batch >= 1 && max_batch <= 4096, "max_batch must be 1..4096");
  kf_prior* P = new kf_prior();
  P->max_batch = max_batch;
  P->nparams = layout().total;
  const long B = max_batch;
  hipError_t e = hipSuccess;
  auto al = [&](void** p, size_t bytes) {
    if (e == hipSuccess) e = hipMalloc(p, bytes);
  };
  al((void**)&P->params, P->nparams * 4);
  al((void**)&P->wbf, P->nparams * 2);
  al((void**)&P->wt, weight_copies().total * 2);
  al((void**)&P->grad, P->nparams * 4);
  al((void**)&P->adam_m, P->nparams * 4);
  al((void**)&P->adam_v, P->nparams * 4);
  for (int l = 0; l < kConvs; ++l) {
    const ConvShape& c = kConv[l];
    const long M = B * c.hout * c.wout;
    if (l + 1 < kConvs) {
      al((void**)&P->Yb[l], M * c.cout * 2);
      al((void**)&P->signs[l], M * c.cout / 8);
    }
    else al((void**)&P->Y4, M * c.cout * 4);
    al((void**)&P->wpart[l], (l == 0 ? kDgradMore : kWgradBlocks / (c.cout / (l == 1 ? 64 : 32))) * c.cout * c.kc * 4);
    if (l > 0) al((void**)&P->dYb[l], M * c.cout * 2);  // layer 1's stays in the kernel that makes it
    al((void**)&P->bpart[l], (l + 1 < kConvs ? kDgradMore : B) * c.cout * 4);
  }
  al((void**)&P->X5b, B * kX5Pitch * 2);
  al((void**)&P->Hb, B * kHidden * 2);
  al((void**)&P->O, B * kTwist * 4);
  al((void**)&P->dO, B * kDoSumPitch * 4);
  al((void**)&P->dOb, B * kDoPitch * 2);
  al((void**)&P->dH, B * kHidden * 4);
  al((void**)&P->dHb, B * kHidden * 2);
  al((void**)&P->fuse_count, B * sizeof(unsigned));
  if (e == hipSuccess) e = hipMemset(P->fuse_count, 0, B * sizeof(unsigned));
  if (e == hipSuccess) e = hipMemset(P->wt, 0, weight_copies().total * 2);  // the copies' padding
  if (e == hipSuccess) e = hipMemset(P->adam_m, 0, P->nparams * 4);
  if (e == hipSuccess) e = hipMemset(P->adam_v, 0, P->nparams * 4);
  if (e == hipSuccess) e = hipMemset(P->params, 0, P->nparams * 4);
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e != hipSuccess) {
    kf_prior_destroy(P);
    return hip_fail(e, "prior allocation");
  }
  *out = P;
  return KF_OK;
}

extern "C" kf_status kf_prior_set_params(kf_prior* P, const float* h, int64_t count) {
  KF_CHECK_ARG(P && h, "NULL argument");
  KF_CHECK_ARG(count == P->nparams, "parameter count mismatch");
  KF_HIP(hipMemcpy(P->params, h, count * 4, hipMemcpyHostToDevice));
  KF_TRY(sync_weights(P, nullptr));
  KF_HIP(hipDeviceSynchronize());
  return KF_OK;
}

extern "C" kf_status kf_prior_get_params(kf_prior* P, float* h, int64_t count) {
  KF_CHECK_ARG(P && h, "NULL argument");
  KF_CHECK_ARG(count == P->nparams, "parameter count mismatch");
  KF_HIP(hipDeviceSynchronize());
  KF_HIP(hipMemcpy(h, P->params, count * 4, hipMemcpyDeviceToHost));
  return KF_OK;
}

extern "C" kf_status kf_prior_init_params(kf_prior* P, uint64_t seed) {
  KF_CHECK_ARG(P != nullptr, "NULL argument");
  const ParamLayout& L = layout();
  std::vector<float> h(P->nparams, 0.0f);
  uint64_t st = seed * 0x9E3779B97F4A7C15ull + 0x1234567ull;
  auto uni = [&]() {
    st ^= st << 13;
    st ^= st >> 7;
    st ^= st << 17;
    return (double)(st >> 11) * (1.0 / 9007199254740992.0);
  };
  const long fan_in[6] = {kConv[0].kc, kConv[1].kc, kConv[2].kc, kConv[3].kc, kFc1In, kHidden};
  for (int l = 0; l < 6; ++l) {
    const long n = L.b[l] - L.w[l];
    const double a = sqrt(6.0 / (double)fan_in[l]) * (l == 5 ? 0.1 : 1.0);
    for (long i = 0; i < n; ++i) h[L.w[l] + i] = (float)((2.0 * uni() - 1.0) * a);
  }
  KF_TRY(kf_prior_set_params(P, h.data(), P->nparams));
  KF_HIP(hipMemset(P->adam_m, 0, P->nparams * 4));
  KF_HIP(hipMemset(P->adam_v, 0, P->nparams * 4));
  P->step = 0;
  return KF_OK;
}

extern "C" kf_status kf_prior_forward(kf_prior* P, const float* frames, const int32_t* pairs, const float* prev,
                                      int32_t B, float* d_out, kf_stream s) {
  KF_TRY(check_batch(P, frames, pairs, prev, B));
  KF_CHECK_ARG(d_out != nullptr, "out is NULL");
  return infer(P, frames, pairs, prev, B, d_out, S(s));
}

extern "C" kf_status kf_prior_gradients(kf_prior* P, const float* frames, const int32_t* pairs, const float* prev,
                                        const float* target, int32_t B, float* d_grad, float* d_loss, kf_stream s) {
  KF_TRY(check_batch(P, frames, pairs, prev, B));
  KF_CHECK_ARG(target && d_grad, "NULL argument");
  KF_TRY(forward(P, frames, pairs, B, true, S(s)));
  return backward(P, frames, pairs, prev, target, B, d_grad, d_loss, S(s));
}

extern "C" kf_status kf_prior_train_step(kf_prior* P, const float* frames, const int32_t* pairs, const float* prev,
                                         const float* target, int32_t B, float lr, float* d_loss, kf_stream s) {
  KF_TRY(check_batch(P, frames, pairs, prev, B));
  KF_CHECK_ARG(target != nullptr, "target is NULL");
  KF_TRY(forward(P, frames, pairs, B, true, S(s)));
  KF_TRY(backward(P, frames, pairs, prev, target, B, P->grad, d_loss, S(s)));
  P->step += 1;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.0f - (float)pow(0.9, (double)P->step), c2 = 1.0f - (float)pow(0.999, (double)P->step);
  hipLaunchKernelGGL(adam, dim3(blocks_for(P->nparams)), dim3(256), 0, S(s), copy_args(P), P->params,
                     (const float*)P->grad, P->adam_m, P->adam_v, P->nparams, lr, b1, b2, 1e-8f, c1, c2);
  return check_launch("adam");
}
