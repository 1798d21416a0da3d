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
// the maps directly (kf_prior_conv.hpp).  The fully connected layers' GEMM is one 16x16
// output tile per wavefront on v_mfma_f32_16x16x32_bf16, four wavefronts per 256-thread
// block.
#include "kf_prior_conv.hpp"

#include <math.h>
#include <string.h>

#include <algorithm>
#include <vector>

namespace kf {
namespace {

// ---------------------------------------------------------------------------
// GEMM: C[m][n] (+)= sum_k A(m,k) B(k,n); A(m,k) = A[m*sam + k*sak], B(k,n) =
// B[k*sbk + n*sbn] (BF16 bits).
struct GemmArgs {
  const uint16_t* A;
  long sam, sak;
  const uint16_t* B;
  long sbk, sbn;
  float* C;
  long ldc;
  int M, N, K, accumulate;
  // Epilogue: v = acc [+ bias[n], ReLU] [+ addend[m * N + n]]; C = v and,
  // with Cb, the BF16 copy (RNE) at the same position.
  const float* bias;
  int relu;
  const float* addend;
  uint16_t* Cb;
};

// Each 256-thread block computes a 32x32 tile of C (four 16x16 wave tiles on
// v_mfma_f32_16x16x32_bf16).  K is staged through LDS in chunks of kKc: the block
// loads the 32 x chunk slices of A and B with coalesced accesses (adjacent threads
// take adjacent addresses along whichever of K or M/N is unit-stride), then runs
// the chunk's MFMAs from LDS, each operand one 16-byte LDS read per lane.  The MFMA
// sequence over k (steps of 32 from 0, zeros beyond K) is the same as a direct k
// loop, so results do not depend on the chunking; any kernel that runs the same
// sequence on the same operands gets the same bits.
constexpr int kKc = 576;        // K per chunk
constexpr int kPitch = kKc + 8;  // LDS row pitch (elements): rows start on different banks
constexpr int kVecPerThread = (32 * kKc / 8 + 255) / 256;  // 16-byte vectors per thread and operand

// Stages a 32 x kpad operand slice into T[32][kPitch] (row = m or n, column = k)
// from X(row, k) = X[row * s_row + k * s_k], zero outside rows < nrows, k < kn.
__device__ __forceinline__ void stage(uint16_t (*T)[kPitch], const uint16_t* X, long s_row, long s_k, int row0,
                                      int nrows, long k0, int kn, int kpad) {
  const int tid = threadIdx.x;
  const bool vec = s_k == 1 && (s_row & 7) == 0 && (k0 & 7) == 0 && (kn & 7) == 0 &&
                   ((reinterpret_cast<uintptr_t>(X) & 15) == 0);
  if (vec) {  // 16-byte loads of 8 consecutive k, all issued before any LDS store
    const int vpr = kpad >> 3;  // vectors per row (the last one may be k padding)
    const int total = 32 * vpr;
    uint4 v[kVecPerThread];
#pragma unroll
    for (int u = 0; u < kVecPerThread; ++u) {
      const int e = tid + 256 * u;
      const int r = e / vpr, c = e - (e / vpr) * vpr;
      const bool in = e < total && row0 + r < nrows && 8 * c < kn;
      v[u] = in ? *reinterpret_cast<const uint4*>(X + (long)(row0 + r) * s_row + k0 + 8 * c) : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < kVecPerThread; ++u) {
      const int e = tid + 256 * u;
      if (e < total) {
        const int r = e / vpr, c = e - (e / vpr) * vpr;
        *reinterpret_cast<uint4*>(&T[r][8 * c]) = v[u];
      }
    }
  } else if (s_k == 1) {  // K contiguous: thread e takes (row, k) = (e / kpad, e % kpad)
    const int total = 32 * kpad;
    for (int e0 = tid; e0 < total; e0 += 256 * 4) {
      uint16_t v[4];
      int rr[4], kk[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int e = e0 + 256 * u;
        rr[u] = e / kpad;
        kk[u] = e - rr[u] * kpad;
        const bool in = e < total && row0 + rr[u] < nrows && kk[u] < kn;
        v[u] = in ? X[(long)(row0 + rr[u]) * s_row + (k0 + kk[u])] : (uint16_t)0;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (e0 + 256 * u < total) T[rr[u]][kk[u]] = v[u];
    }
  } else {  // rows contiguous (or general): thread e takes (k, row) = (e / 32, e % 32)
    const int total = 32 * kpad;
    for (int e0 = tid; e0 < total; e0 += 256 * 4) {
      uint16_t v[4];
      int rr[4], kk[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int e = e0 + 256 * u;
        kk[u] = e >> 5;
        rr[u] = e & 31;
        const bool in = e < total && row0 + rr[u] < nrows && kk[u] < kn;
        v[u] = in ? X[(long)(row0 + rr[u]) * s_row + (k0 + kk[u]) * s_k] : (uint16_t)0;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (e0 + 256 * u < total) T[rr[u]][kk[u]] = v[u];
    }
  }
}

__global__ __launch_bounds__(256) void gemm_bf16(GemmArgs g) {
  __shared__ __align__(16) uint16_t As[32][kPitch];
  __shared__ __align__(16) uint16_t Bt[32][kPitch];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int mt = blockIdx.y * 32, nt = blockIdx.x * 32;
  const int wm = (wave >> 1) * 16, wn = (wave & 1) * 16;
  const int r = lane & 15, kq = (lane >> 4) * 8;
  v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int kc0 = 0; kc0 < g.K; kc0 += kKc) {
    const int kn = min(kKc, g.K - kc0);
    const int kpad = (kn + 31) & ~31;
    stage(As, g.A, g.sam, g.sak, mt, g.M, kc0, kn, kpad);
    stage(Bt, g.B, g.sbn, g.sbk, nt, g.N, kc0, kn, kpad);
    __syncthreads();
    for (int kk = 0; kk < kpad; kk += 32)
      acc = mfma32(*reinterpret_cast<const uint4*>(&As[wm + r][kk + kq]),
                   *reinterpret_cast<const uint4*>(&Bt[wn + r][kk + kq]), acc);
    __syncthreads();
  }
  const int m0 = mt + wm, n0 = nt + wn;
  if (m0 >= g.M || n0 >= g.N) return;  // wave-uniform
  const int cn = n0 + (lane & 15);
  if (cn >= g.N) return;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int cm = m0 + (lane >> 4) * 4 + j;
    if (cm >= g.M) continue;
    {
      float* c = g.C + (long)cm * g.ldc + cn;
      float v = g.accumulate ? *c + acc[j] : acc[j];
      if (g.bias) {
        v = v + g.bias[cn];
        if (g.relu) v = fmaxf(v, 0.0f);
      }
      if (g.addend) v = v + g.addend[(long)cm * g.N + cn];
      *c = v;
      if (g.Cb) g.Cb[(long)cm * g.ldc + cn] = bf16_rne(v);
    }
  }
}

// ---------------------------------------------------------------------------
// Fused inference (kf_prior_forward): one 256-thread block per (layer-4 pixel,
// sample) carries the pixel's receptive field through the four convolutions in
// LDS — a 15x15 window of layer 1, 7x7 of layer 2, 3x3 of layer 3, then the pixel
// (window positions outside a layer's map hold zeros: that layer's padding) — and
// computes every output with the MFMA sequence gemm_bf16 runs for it (k steps of
// 32 from 0 on the same BF16 operands, the same epilogue), so every activation
// equals the layer-by-layer forward's bit for bit.  Neighbouring blocks recompute
// the overlap of their windows (~2.7x the 42 M MACs of one sample) in exchange for
// one launch instead of eight, with nothing between the layers but LDS.  The last
// block of a sample to finish (a device counter, cleared again by that block)
// averages the 80 layer-4 pixels and runs FC1 and FC2 for the sample's row as
// gemm_bf16 would.  Operands: A from LDS and B (weights, L2-resident) from global
// memory, one 16-byte vector per lane and MFMA step.
constexpr int kFuseThreads = 256;
constexpr int kWin1 = 15, kWin2 = 7, kWin3 = 3;  // window sides of layers 1-3 around one layer-4 pixel
constexpr int kRows1 = kWin1 * kWin1;            // 225 layer-1 positions
constexpr int kRows1Pad = 240;                   // 15 MFMA row tiles
constexpr int kFc1Pad = 160;                     // FC1 K (134) rounded up to the MFMA step
constexpr int kPatch = 2 * kWin1 + 1;            // 31: input window side

struct FuseArgs {
  const float* frames;
  const int32_t* pairs;
  const float* prev;
  const uint16_t* wbf;   // BF16 weights
  const float* params;   // FP32 biases
  long w[6], b[6];       // parameter offsets
  float* Y4;             // [B][80][128] layer-4 activations
  float* X5;             // [B][134] pooled features and previous twist
  uint16_t* X5b;
  float* H;              // [B][256] FC1 output
  uint16_t* Hb;
  float* out;            // [B][6]
  unsigned* count;       // [B] finished blocks of each sample (zero between calls)
};

// B operand of one MFMA step for output column n: W(n, k .. k + 7) of the row-major
// [N][kc] BF16 weights, zero for n >= N or beyond kc.
__device__ __forceinline__ uint4 wfrag(const uint16_t* W, int kc, int N, int n, int k) {
  if (n >= N || k >= kc) return make_uint4(0u, 0u, 0u, 0u);
  const uint16_t* row = W + (long)n * kc;
  if ((kc & 7) == 0) return *reinterpret_cast<const uint4*>(row + k);  // 16-byte aligned rows
  uint16_t e[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) e[j] = k + j < kc ? row[k + j] : (uint16_t)0;
  uint4 r;
  __builtin_memcpy(&r, e, 16);
  return r;
}

// A operand of one MFMA step of a 3x3 / stride-2 convolution over an LDS window of
// side 2 WOUT + 1 (NHWC, CIN channels): output window position p, k .. k + 7 = eight
// channels of one tap.
template <int CIN, int WOUT>
__device__ __forceinline__ uint4 afrag(const uint16_t* act, int p, int k) {
  const int tap = k / CIN, ci = k - tap * CIN;
  const int ky = tap / 3, kx = tap - 3 * ky;
  const int wy = p / WOUT, wx = p - wy * WOUT;
  return *reinterpret_cast<const uint4*>(act + ((2 * wy + ky) * (2 * WOUT + 1) + (2 * wx + kx)) * CIN + ci);
}

// One convolution layer of the window (layers 2-4): output window side WOUT with
// origin (y0, x0) in a map of HOUT x WOUT_MAP; wave w takes column tiles w, w + 4,
// ... and every row tile.  Epilogue as gemm_bf16's (bias, ReLU); layers 2-3 store
// the BF16 copy into the output window (zero outside the map), layer 4 (WOUT 1)
// stores the FP32 value of its one position to y4.
template <int CIN, int COUT, int WOUT, int HOUT, int WOUT_MAP>
__device__ __forceinline__ void fuse_conv(const uint16_t* in, uint16_t* outw, const uint16_t* W, const float* bias,
                                          int y0, int x0, float* y4) {
  constexpr int K = 9 * CIN, STEPS = K / 32, ROWS = WOUT * WOUT, MT = (ROWS + 15) / 16, NT = COUT / 16;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, q = lane >> 4;
  for (int nt = wave; nt < NT; nt += kFuseThreads / kWave) {
    const int n = nt * 16 + r;
    uint4 bf[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) bf[s] = wfrag(W, K, COUT, n, 32 * s + 8 * q);
    const float bn = bias[n];
    for (int mt = 0; mt < MT; ++mt) {
      const int p = min(mt * 16 + r, ROWS - 1);  // rows beyond the window repeat the last one
      v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int s = 0; s < STEPS; ++s) acc = mfma32(afrag<CIN, WOUT>(in, p, 32 * s + 8 * q), bf[s], acc);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int row = mt * 16 + 4 * q + j;
        if (row >= ROWS) continue;
        float v = acc[j] + bn;
        v = fmaxf(v, 0.0f);
        if (y4) {
          if (row == 0) y4[n] = v;
        } else {
          const int wy = row / WOUT, wx = row - wy * WOUT;
          const int gy = y0 + wy, gx = x0 + wx;
          const bool in_map = gy >= 0 && gy < HOUT && gx >= 0 && gx < WOUT_MAP;
          outw[row * COUT + n] = in_map ? bf16_rne(v) : (uint16_t)0;
        }
      }
    }
  }
}

__global__ __launch_bounds__(kFuseThreads) void prior_infer_fused(FuseArgs f) {
  __shared__ uint16_t patch[2][kPatch][kPatch];              // input window (two planes), BF16
  __shared__ __align__(16) uint16_t col1[kRows1Pad * 32];    // layer-1 im2col of the window
  __shared__ __align__(16) uint16_t act1[kRows1 * 32];       // layer-1 window, NHWC
  __shared__ __align__(16) uint16_t act2[kWin2 * kWin2 * 64];
  __shared__ __align__(16) uint16_t act3[kWin3 * kWin3 * 64];
  __shared__ __align__(16) uint16_t xs[kFc1Pad];
  __shared__ __align__(16) uint16_t hs[kHidden];
  __shared__ int s_last;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, q = lane >> 4;
  const int n = blockIdx.y, pix = blockIdx.x;
  const int y4 = pix / kConv[3].wout, x4 = pix - y4 * kConv[3].wout;
  const int f0 = f.pairs[2 * n], f1 = f.pairs[2 * n + 1];

  // the 31x31 input window of both planes (zero outside the frame), BF16 as im2col_pairs rounds it
  {
    constexpr int E = 2 * kPatch * kPatch, PER = (E + kFuseThreads - 1) / kFuseThreads;
    float v[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int e = tid + kFuseThreads * u;
      const int c = e / (kPatch * kPatch), rem = e - c * (kPatch * kPatch);
      const int py = rem / kPatch, px = rem - py * kPatch;
      const int iy = 16 * y4 - 15 + py, ix = 16 * x4 - 15 + px;
      const bool in = e < E && iy >= 0 && iy < kH0 && ix >= 0 && ix < kW0;
      v[u] = in ? f.frames[((long)(c ? f1 : f0) * kH0 + iy) * kW0 + ix] : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int e = tid + kFuseThreads * u;
      if (e < E) {
        const int c = e / (kPatch * kPatch), rem = e - c * (kPatch * kPatch);
        const int py = rem / kPatch, px = rem - py * kPatch;
        patch[c][py][px] = bf16_rne(v[u]);
      }
    }
  }
  __syncthreads();
  // layer-1 im2col of the 15x15 window (k = (ky * 3 + kx) * 2 + plane, zero for k >= 18)
  for (int e = tid; e < kRows1Pad * 32; e += kFuseThreads) {
    const int p = e >> 5, k = e & 31;
    uint16_t v = 0;
    if (p < kRows1 && k < kConv[0].kc) {
      const int wy = p / kWin1, wx = p - wy * kWin1;
      const int tap = k >> 1, ky = tap / 3, kx = tap - 3 * ky;
      v = patch[k & 1][2 * wy + ky][2 * wx + kx];
    }
    col1[e] = v;
  }
  __syncthreads();
  // layer 1: M = 225 window positions, N = 32, one K step; wave w: column tile w & 1,
  // row tiles (w >> 1), (w >> 1) + 2, ...
  {
    const int nt = wave & 1, nn = nt * 16 + r;
    const uint4 bw = wfrag(f.wbf + f.w[0], kConv[0].kc, 32, nn, 8 * q);
    const float bn = f.params[f.b[0] + nn];
    for (int mt = wave >> 1; mt < kRows1Pad / 16; mt += 2) {
      const uint4 a = *reinterpret_cast<const uint4*>(&col1[(mt * 16 + r) * 32 + 8 * q]);
      v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
      acc = mfma32(a, bw, acc);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int row = mt * 16 + 4 * q + j;
        if (row >= kRows1) continue;
        const float v = fmaxf(acc[j] + bn, 0.0f);
        const int wy = row / kWin1, wx = row - wy * kWin1;
        const int gy = 8 * y4 - 7 + wy, gx = 8 * x4 - 7 + wx;
        const bool in_map = gy >= 0 && gy < kConv[0].hout && gx >= 0 && gx < kConv[0].wout;
        act1[row * 32 + nn] = in_map ? bf16_rne(v) : (uint16_t)0;
      }
    }
  }
  __syncthreads();
  fuse_conv<32, 64, kWin2, 30, 40>(act1, act2, f.wbf + f.w[1], f.params + f.b[1], 4 * y4 - 3, 4 * x4 - 3, nullptr);
  __syncthreads();
  fuse_conv<64, 64, kWin3, 15, 20>(act2, act3, f.wbf + f.w[2], f.params + f.b[2], 2 * y4 - 1, 2 * x4 - 1, nullptr);
  __syncthreads();
  float* y4row = f.Y4 + ((long)n * kPool + pix) * kFeat;
  fuse_conv<64, 128, 1, 8, 10>(act3, nullptr, f.wbf + f.w[3], f.params + f.b[3], y4, x4, y4row);

  // the last block of the sample: every other block's layer-4 pixel is visible to it
  __builtin_amdgcn_s_waitcnt(0);  // this thread's stores have completed
  __syncthreads();
  if (tid == 0) {
    __threadfence();
    const unsigned done = atomicAdd(&f.count[n], 1u);
    s_last = done == (unsigned)(kPool - 1);
    if (s_last) __threadfence();
  }
  __syncthreads();
  if (!s_last) return;  // uniform

  // pooling and the previous twist (as pool_concat)
  if (tid < kFc1In) {
    float v;
    if (tid < kFeat) {
      float sum = 0.0f;
      for (int p = 0; p < kPool; ++p) sum = sum + f.Y4[((long)n * kPool + p) * kFeat + tid];
      v = sum * (1.0f / (float)kPool);
    } else {
      v = f.prev[n * kTwist + (tid - kFeat)];
    }
    f.X5[n * kFc1In + tid] = v;
    const uint16_t vb = bf16_rne(v);
    f.X5b[n * kFc1In + tid] = vb;
    xs[tid] = vb;
  } else if (tid < kFc1Pad) {
    xs[tid] = 0;
  }
  __syncthreads();
  // FC1 (row n only): H = ReLU(X5 W5^T + b5), K = 134 in 5 steps; wave w: column tiles w, w + 4, ...
  for (int nt = wave; nt < kHidden / 16; nt += kFuseThreads / kWave) {
    const int nn = nt * 16 + r;
    v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < kFc1Pad; k += 32)
      acc = mfma32(*reinterpret_cast<const uint4*>(&xs[k + 8 * q]), wfrag(f.wbf + f.w[4], kFc1In, kHidden, nn, k + 8 * q),
                   acc);
    if (q == 0) {  // row 0: the sample's row
      const float v = fmaxf(acc[0] + f.params[f.b[4] + nn], 0.0f);
      f.H[n * kHidden + nn] = v;
      const uint16_t vb = bf16_rne(v);
      f.Hb[n * kHidden + nn] = vb;
      hs[nn] = vb;
    }
  }
  __syncthreads();
  // FC2 plus the skip connection (one wave): O = (H W6^T + b6) + previous twist
  if (wave == 0) {
    v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < kHidden; k += 32)
      acc = mfma32(*reinterpret_cast<const uint4*>(&hs[k + 8 * q]), wfrag(f.wbf + f.w[5], kHidden, kTwist, r, k + 8 * q),
                   acc);
    if (q == 0 && r < kTwist) {
      float v = acc[0] + f.params[f.b[5] + r];
      v = v + f.prev[n * kTwist + r];
      f.out[n * kTwist + r] = v;
    }
    if (lane == 0) f.count[n] = 0u;  // ready for the next call
  }
}

__global__ void to_bf16(const float* x, uint16_t* y, long n) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = bf16_rne(x[i]);
}

// feat[n][0..127] = mean over the 80 pooled pixels of Y4; [128..133] = prev twist.
__global__ void pool_concat(const float* Y4, const float* prev, int batch, float* X5, uint16_t* X5b) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= batch * kFc1In) return;
  const int n = i / kFc1In, c = i - n * kFc1In;
  float v;
  if (c < kFeat) {
    float s = 0.0f;
    for (int p = 0; p < kPool; ++p) s = s + Y4[((long)n * kPool + p) * kFeat + c];
    v = s * (1.0f / (float)kPool);
  } else {
    v = prev[n * kTwist + (c - kFeat)];
  }
  X5[i] = v;
  X5b[i] = bf16_rne(v);
}

// BF16 copies of the parameters: y in the blob's order, and the weights of layers 2-4
// again as [tap][ci][co] (yt, at the blob's offsets) for the input gradients.
struct WeightCopyArgs {
  const float* x;
  uint16_t *y, *yt;
  long n, w[kConvs];  // parameter count, weight offsets of the convolutions
};
__global__ void copy_weights(WeightCopyArgs a) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  const uint16_t v = bf16_rne(a.x[i]);
  a.y[i] = v;
#pragma unroll
  for (int l = 1; l < kConvs; ++l) {
    const int e = (int)(i - a.w[l]);
    if (e >= 0 && e < kConv[l].cout * kConv[l].kc) a.yt[a.w[l] + (e % kConv[l].kc) * kConv[l].cout + e / kConv[l].kc] = v;
  }
}

// dY4[n][p][c] = dX5[n][c] / 80 where Y4 > 0, as BF16, and each sample's FP32 sums over
// its pixels (bpart[n][c]).  One block per sample.
__global__ __launch_bounds__(2 * kFeat) void pool_backward(const float* dX5, const float* Y4, uint16_t* dY4, float* bpart) {
  __shared__ float red[kFeat];
  const int n = blockIdx.x, c = threadIdx.x & (kFeat - 1), half = threadIdx.x / kFeat;
  const float g = dX5[n * kFc1In + c] * (1.0f / (float)kPool);
  float s = 0.0f;
#pragma unroll 8
  for (int p = half; p < kPool; p += 2) {
    const long i = ((long)n * kPool + p) * kFeat + c;
    const float v = Y4[i] > 0.0f ? g : 0.0f;
    dY4[i] = bf16_rne(v);
    s = s + v;
  }
  if (half == 1) red[c] = s;
  __syncthreads();
  if (half == 0) bpart[(long)n * kFeat + c] = s + red[c];
}

// Loss mean((O - T)^2) and dO = 2 (O - T) / (6 B); one block.
__global__ void mse_loss(const float* O, const float* T, int batch, float* dO, float* loss) {
  __shared__ float red[256];
  const int n = batch * kTwist;
  const float inv = 1.0f / (float)n;
  float s = 0.0f;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const float d = O[i] - T[i];
    dO[i] = 2.0f * d * inv;
    s = s + d * d;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0 && loss) *loss = red[0] * inv;
}

// db[c] = sum_m dY[m][c]; one block per channel, fixed reduction order.
__global__ void bias_grad(const float* dY, long M, int C, float* db) {
  __shared__ float red[256];
  const int c = blockIdx.x;
  float s = 0.0f;
  for (long m = threadIdx.x; m < M; m += blockDim.x) s = s + dY[m * C + c];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) db[c] = red[0];
}

__global__ void relu_mask(float* dY, const float* Y, long n) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && !(Y[i] > 0.0f)) dY[i] = 0.0f;
}

__global__ void adam(float* p, const float* g, float* m, float* v, long n, float lr, float b1, float b2, float eps,
                     float c1, float c2) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

inline unsigned blocks_for(long n, int t = 256) { return (unsigned)((n + t - 1) / t); }

}  // namespace
}  // namespace kf

struct kf_prior {
  int max_batch = 0;
  long nparams = 0;
  float* params = nullptr;   // FP32 master
  uint16_t* wbf = nullptr;   // BF16 copy
  uint16_t* wt = nullptr;    // layers 2-4 again as [tap][ci][co], at the same offsets
  float* grad = nullptr;
  float* adam_m = nullptr;
  float* adam_v = nullptr;
  long step = 0;
  // activations (NHWC), sized for max_batch
  uint16_t* Yb[kf::kConvs - 1] = {};  // layers 1-3, BF16 NHWC
  float* Y4 = nullptr;                // layer 4, FP32
  float* X5 = nullptr;
  uint16_t* X5b = nullptr;
  float* Hd = nullptr;
  uint16_t* Hb = nullptr;
  float* O = nullptr;
  float* dO = nullptr;
  uint16_t* dOb = nullptr;
  float* dH = nullptr;
  uint16_t* dHb = nullptr;
  float* dX5 = nullptr;
  uint16_t* dYb[kf::kConvs] = {};       // gradients of the layers' outputs, BF16 NHWC
  float* bpart[kf::kConvs] = {};        // partial bias sums per block (layer 4: per sample)
  float* wpart[kf::kConvs] = {};        // partial weight gradients per split
  float* loss_tmp = nullptr;
  unsigned* fuse_count = nullptr;  // [max_batch] finished blocks per sample of the fused inference
};

namespace kf {
namespace {

struct Epilogue {
  const float* bias = nullptr;
  int relu = 0;
  const float* addend = nullptr;
  uint16_t* Cb = nullptr;
};

kf_status gemm(hipStream_t s, const uint16_t* A, long sam, long sak, const uint16_t* B, long sbk, long sbn, float* C,
               long ldc, int M, int N, int K, bool accumulate,
               const Epilogue& ep = Epilogue()) {
  GemmArgs g;
  g.bias = ep.bias;
  g.relu = ep.relu;
  g.addend = ep.addend;
  g.Cb = ep.Cb;
  g.A = A;
  g.sam = sam;
  g.sak = sak;
  g.B = B;
  g.sbk = sbk;
  g.sbn = sbn;
  g.C = C;
  g.ldc = ldc;
  g.M = M;
  g.N = N;
  g.K = K;
  g.accumulate = accumulate ? 1 : 0;
  dim3 grid((N + 31) / 32, (M + 31) / 32);
  hipLaunchKernelGGL(gemm_bf16, grid, dim3(256), 0, s, g);
  KF_TRY(check_launch("gemm_bf16"));
  return KF_OK;
}

// BF16 copies of the weights; every call that changes the FP32 parameters refreshes
// them, so inference (forward) never converts.
kf_status sync_weights(kf_prior* P, hipStream_t s) {
  WeightCopyArgs a;
  a.x = P->params;
  a.y = P->wbf;
  a.yt = P->wt;
  a.n = P->nparams;
  for (int l = 0; l < kConvs; ++l) a.w[l] = layout().w[l];
  hipLaunchKernelGGL(copy_weights, dim3(blocks_for(P->nparams)), dim3(256), 0, s, a);
  return check_launch("copy_weights");
}

// Inference: the fused kernel (the training forward's outputs, in one launch).
kf_status infer(kf_prior* P, const float* frames, const int32_t* pairs, const float* prev, int B, float* out,
                hipStream_t s) {
  const ParamLayout& L = layout();
  FuseArgs f;
  f.frames = frames;
  f.pairs = pairs;
  f.prev = prev;
  f.wbf = P->wbf;
  f.params = P->params;
  for (int q = 0; q < 6; ++q) {
    f.w[q] = L.w[q];
    f.b[q] = L.b[q];
  }
  f.Y4 = P->Y4;
  f.X5 = P->X5;
  f.X5b = P->X5b;
  f.H = P->Hd;
  f.Hb = P->Hb;
  f.out = out;
  f.count = P->fuse_count;
  hipLaunchKernelGGL(prior_infer_fused, dim3(kPool, B), dim3(kFuseThreads), 0, s, f);
  return check_launch("prior_infer_fused");
}

constexpr int kConvBlocks = 512;

// One convolution of the training forward: two blocks of four waves a CU hold the
// weights; a small batch gets one wave per 16-pixel tile and channel group.
template <int L, int NT, bool F32>
kf_status launch_conv(kf_prior* P, const uint16_t* X, uint16_t* Yb, float* Y, int B, hipStream_t s) {
  constexpr ConvShape c = kConv[L];
  constexpr int GROUPS = c.cout / (16 * NT);
  const ParamLayout& lay = layout();
  const int M = B * c.hout * c.wout;
  const int blocks = std::min(div_up(div_up(M, 16) * GROUPS, kConvWaves), kConvBlocks);
  hipLaunchKernelGGL((conv_forward<L, NT, F32>), dim3(blocks), dim3(kConvThreads), 0, s, X, P->wbf + lay.w[L],
                     (const float*)P->params + lay.b[L], Yb, Y, M);
  return check_launch("conv_forward");
}

// Training forward: the activations stay for the backward pass.
kf_status forward(kf_prior* P, const float* frames, const int32_t* pairs, const float* prev, int B, hipStream_t s) {
  const ParamLayout& L = layout();
  hipLaunchKernelGGL(conv1_forward, dim3(kConv[0].hout / kL1Rows, B), dim3(kConvThreads), 0, s, frames, pairs,
                     (const uint16_t*)P->wbf + L.w[0], (const float*)P->params + L.b[0], P->Yb[0]);
  KF_TRY(check_launch("conv1_forward"));
  KF_TRY((launch_conv<1, 4, false>(P, P->Yb[0], P->Yb[1], nullptr, B, s)));
  KF_TRY((launch_conv<2, 2, false>(P, P->Yb[1], P->Yb[2], nullptr, B, s)));
  KF_TRY((launch_conv<3, 2, true>(P, P->Yb[2], nullptr, P->Y4, B, s)));
  hipLaunchKernelGGL(pool_concat, dim3(blocks_for((long)B * kFc1In)), dim3(256), 0, s, (const float*)P->Y4, prev, B,
                     P->X5, P->X5b);
  KF_TRY(check_launch("pool_concat"));
  {  // FC1: H = ReLU(X5 W5^T + b5), also as BF16 for FC2
    Epilogue ep;
    ep.bias = (const float*)P->params + L.b[4];
    ep.relu = 1;
    ep.Cb = P->Hb;
    KF_TRY(gemm(s, P->X5b, kFc1In, 1, P->wbf + L.w[4], 1, kFc1In, P->Hd, kHidden, B, kHidden, kFc1In, false, ep));
  }
  {  // FC2 plus the skip connection: O = (H W6^T + b6) + previous twist
    Epilogue ep;
    ep.bias = (const float*)P->params + L.b[5];
    ep.addend = prev;
    KF_TRY(gemm(s, P->Hb, kHidden, 1, P->wbf + L.w[5], 1, kHidden, P->O, kTwist, B, kTwist, kHidden,
                false, ep));
  }
  return KF_OK;
}

// Input gradient of layer L (dYb[L] -> dYb[L - 1], partial sums of layer L - 1's bias
// gradient; *planes: how many), on the grid of launch_conv.
template <int L, int NT>
kf_status launch_dgrad(kf_prior* P, int B, int* planes, hipStream_t s) {
  constexpr ConvShape c = kConv[L];
  const int M = B * c.hout * c.wout;
  *planes = std::min(div_up(div_up(M, 16) * (c.cin / (16 * NT)), kConvWaves), kConvBlocks);
  hipLaunchKernelGGL((conv_dgrad<L, NT>), dim3(*planes), dim3(kConvThreads), 0, s, (const uint16_t*)P->dYb[L],
                     (const uint16_t*)P->wt + layout().w[L], (const uint16_t*)P->Yb[L - 1], P->dYb[L - 1],
                     P->bpart[L - 1], M);
  return check_launch("conv_dgrad");
}

// Weight gradient of layer L as *splits partial planes: one block a CU, at least
// kWgradMinSteps steps of 32 pixels each (a shorter split would mostly write its plane).
constexpr int kWgradBlocks = 256, kWgradMinSteps = 4;
template <int L>
kf_status launch_wgrad(kf_prior* P, int B, int* splits, hipStream_t s) {
  constexpr int GROUPS = WgradShape<L>::GROUPS;
  const int M = B * kConv[L].hout * kConv[L].wout, steps = div_up(M, kWgradStep);
  const int want = std::min(std::max(steps / kWgradMinSteps, 1), kWgradBlocks / GROUPS);
  const int per = div_up(steps, want);
  *splits = div_up(steps, per);
  // eight splits a round (blocks of one split on one XCD): the grid is rounded up, and
  // the splits past the last write zero planes that nothing reads
  const int grid = div_up(*splits, 8) * 8 * GROUPS;
  hipLaunchKernelGGL(conv_wgrad<L>, dim3(grid), dim3(kConvThreads), 0, s, (const uint16_t*)P->dYb[L],
                     (const uint16_t*)P->Yb[L - 1], P->wpart[L], M, per);
  return check_launch("conv_wgrad");
}

kf_status backward(kf_prior* P, const float* frames, const int32_t* pairs, const float* target, int B, float* loss, hipStream_t s) {
  const ParamLayout& L = layout();
  float* G = P->grad;
  hipLaunchKernelGGL(mse_loss, dim3(1), dim3(256), 0, s, (const float*)P->O, target, B, P->dO, loss);
  hipLaunchKernelGGL(to_bf16, dim3(blocks_for((long)B * kTwist)), dim3(256), 0, s, (const float*)P->dO, P->dOb,
                     (long)B * kTwist);
  KF_TRY(check_launch("mse_loss"));
  // FC2: dW6[j][k] = sum_n dO[n][j] H[n][k]; db6; dH = dO W6, masked by H > 0.
  KF_TRY(gemm(s, P->dOb, 1, kTwist, P->Hb, kHidden, 1, G + L.w[5], kHidden, kTwist, kHidden, B, false));
  hipLaunchKernelGGL(bias_grad, dim3(kTwist), dim3(256), 0, s, (const float*)P->dO, (long)B, kTwist, G + L.b[5]);
  KF_TRY(gemm(s, P->dOb, kTwist, 1, P->wbf + L.w[5], kHidden, 1, P->dH, kHidden, B, kHidden, kTwist, false));
  hipLaunchKernelGGL(relu_mask, dim3(blocks_for((long)B * kHidden)), dim3(256), 0, s, P->dH, (const float*)P->Hd,
                     (long)B * kHidden);
  hipLaunchKernelGGL(to_bf16, dim3(blocks_for((long)B * kHidden)), dim3(256), 0, s, (const float*)P->dH, P->dHb,
                     (long)B * kHidden);
  // FC1: dW5[j][k] = sum_n dH[n][j] X5[n][k]; db5; dX5 (features only) = dH W5.
  KF_TRY(gemm(s, P->dHb, 1, kHidden, P->X5b, kFc1In, 1, G + L.w[4], kFc1In, kHidden, kFc1In, B, false));
  hipLaunchKernelGGL(bias_grad, dim3(kHidden), dim3(256), 0, s, (const float*)P->dH, (long)B, kHidden, G + L.b[4]);
  KF_TRY(gemm(s, P->dHb, kHidden, 1, P->wbf + L.w[4], kFc1In, 1, P->dX5, kFc1In, B, kFeat, kHidden, false));
  hipLaunchKernelGGL(pool_backward, dim3(B), dim3(2 * kFeat), 0, s, (const float*)P->dX5, (const float*)P->Y4,
                     P->dYb[3], P->bpart[3]);
  KF_TRY(check_launch("pool_backward"));
  int planes[kConvs] = {0, 0, 0, B}, splits[kConvs];
  KF_TRY(launch_wgrad<3>(P, B, &splits[3], s));
  KF_TRY((launch_dgrad<3, 1>(P, B, &planes[2], s)));
  KF_TRY(launch_wgrad<2>(P, B, &splits[2], s));
  KF_TRY((launch_dgrad<2, 2>(P, B, &planes[1], s)));
  KF_TRY(launch_wgrad<1>(P, B, &splits[1], s));
  KF_TRY((launch_dgrad<1, 2>(P, B, &planes[0], s)));
  const int items = B * (kConv[0].hout / kL1Rows);
  splits[0] = std::min(items, kConvBlocks);
  hipLaunchKernelGGL(conv1_wgrad, dim3(splits[0]), dim3(kConvThreads), 0, s, frames, pairs, (const uint16_t*)P->dYb[0],
                     P->wpart[0], items);
  KF_TRY(check_launch("conv1_wgrad"));
  ReduceArgs red;
  red.jobs = 0;
  red.block0[0] = 0;
  auto add = [&](const float* part, int n, int count, float* out) {
    const int k = red.jobs++;
    red.part[k] = part;
    red.planes[k] = n;
    red.count[k] = count;
    red.out[k] = out;
    red.block0[k + 1] = red.block0[k] + div_up(count, 64);
  };
  for (int l = kConvs - 1; l >= 0; --l) {
    add(P->wpart[l], splits[l], kConv[l].cout * kConv[l].kc, G + L.w[l]);
    add(P->bpart[l], planes[l], kConv[l].cout, G + L.b[l]);
  }
  hipLaunchKernelGGL(reduce_parts, dim3(red.block0[red.jobs]), dim3(1024), 0, s, red);
  KF_TRY(check_launch("reduce_parts"));
  return KF_OK;
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
  void* ptrs[] = {P->params, P->wbf, P->grad, P->adam_m, P->adam_v, P->Y4, P->X5, P->X5b, P->Hd, P->Hb, P->O, P->dO,
                  P->dOb, P->dH, P->dHb, P->dX5, P->wt, P->loss_tmp,
                  P->fuse_count};
  for (void* q : ptrs) (void)hipFree(q);
  for (int l = 0; l < kConvs; ++l) {
    if (l + 1 < kConvs) (void)hipFree(P->Yb[l]);
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
  al((void**)&P->wt, P->nparams * 2);
  al((void**)&P->grad, P->nparams * 4);
  al((void**)&P->adam_m, P->nparams * 4);
  al((void**)&P->adam_v, P->nparams * 4);
  for (int l = 0; l < kConvs; ++l) {
    const ConvShape& c = kConv[l];
    const long M = B * c.hout * c.wout;
    if (l + 1 < kConvs) al((void**)&P->Yb[l], M * c.cout * 2);
    else al((void**)&P->Y4, M * c.cout * 4);
    al((void**)&P->wpart[l], (l == 0 ? kConvBlocks : kWgradBlocks / (c.cout / (l == 1 ? 64 : 32))) * c.cout * c.kc * 4);
    al((void**)&P->dYb[l], M * c.cout * 2);
    al((void**)&P->bpart[l], (l + 1 < kConvs ? kConvBlocks : B) * c.cout * 4);
  }
  al((void**)&P->X5, B * kFc1In * 4);
  al((void**)&P->X5b, B * kFc1In * 2);
  al((void**)&P->Hd, B * kHidden * 4);
  al((void**)&P->Hb, B * kHidden * 2);
  al((void**)&P->O, B * kTwist * 4);
  al((void**)&P->dO, B * kTwist * 4);
  al((void**)&P->dOb, B * kTwist * 2);
  al((void**)&P->dH, B * kHidden * 4);
  al((void**)&P->dHb, B * kHidden * 2);
  al((void**)&P->dX5, B * kFc1In * 4);
  al((void**)&P->loss_tmp, 16);
  al((void**)&P->fuse_count, B * sizeof(unsigned));
  if (e == hipSuccess) e = hipMemset(P->fuse_count, 0, B * sizeof(unsigned));
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
  KF_TRY(forward(P, frames, pairs, prev, B, S(s)));
  KF_TRY(backward(P, frames, pairs, target, B, d_loss, S(s)));
  KF_HIP(hipMemcpyAsync(d_grad, P->grad, (size_t)P->nparams * 4, hipMemcpyDeviceToDevice, S(s)));
  return KF_OK;
}

extern "C" kf_status kf_prior_train_step(kf_prior* P, const float* frames, const int32_t* pairs, const float* prev,
                                         const float* target, int32_t B, float lr, float* d_loss, kf_stream s) {
  KF_TRY(check_batch(P, frames, pairs, prev, B));
  KF_CHECK_ARG(target != nullptr, "target is NULL");
  KF_TRY(forward(P, frames, pairs, prev, B, S(s)));
  KF_TRY(backward(P, frames, pairs, target, B, d_loss, S(s)));
  P->step += 1;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.0f - (float)pow(0.9, (double)P->step), c2 = 1.0f - (float)pow(0.999, (double)P->step);
  hipLaunchKernelGGL(adam, dim3(blocks_for(P->nparams)), dim3(256), 0, S(s), P->params, (const float*)P->grad,
                     P->adam_m, P->adam_v, P->nparams, lr, b1, b2, 1e-8f, c1, c2);
  KF_TRY(check_launch("adam"));
  return sync_weights(P, S(s));
}
