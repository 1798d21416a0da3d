// kf_icp.hip — projective point-to-plane ICP on gfx950, one launch per iteration.
//
// Replaces d_find_corresponding / ICP::FindCorresponding (Source/src/ICP.cu:116-262),
// the host block sum, determinant guard and Eigen LLT of ICP::Iterate_ICP
// (Source/src/ICP.cpp:84-182) and the host pose update of
// ICP::BuildNewTransformMatrix (Source/src/ICP.cu:266-340).
//
// Per model pixel (same association direction and gate structure as the
// reference): the model vertex s / normal m (world) is moved into the live camera
// with the current estimate, projected (round half up), and the live vertex /
// normal there is brought to world (d, n).  The pixel is an inlier iff the live
// depth at the model pixel is valid (ICP.cu:145-149), |d-s| < dist_thresh and
// cos_thresh < n.m < 1+1e-6.  Row: A = [m x d, m], b = m.(s-d); after the solve
// of (A^T A) x = A^T b the rotation is -x[0..2] (ICP.cpp:162-168).
//
// Reduction: 28 terms (21 A^TA, 6 A^Tb, b^2).  In compensated mode they are FP64 (the
// product of two FP32 row entries is exact in FP64): the rows (A, b, inlier flag) of a
// wave's 64 pixels form an 8 x 64 matrix R, and R R^T holds every term and the inlier
// count, so they are sums over pixels on the FP64 matrix cores with no lane reduction
// after them.  Plain mode accumulates FP32 terms per thread and combines waves with DPP
// lane moves (reduce-scatter: row mirrors, quad permutes).  Blocks combine through LDS.
// Each block writes its partial as a slot of FP64 values.  The next launch (the next iteration,
// or the final one-block launch) adds the slots in FP64 in block order, solves by
// FP64 LDL^T and composes the Euler-ZYX increment onto the FP64 pose; every
// block of an iteration repeats that solve for itself, so the pose never makes a
// round trip through the host and an iteration is a single launch.
#include <algorithm>
#include <mutex>

#include "kf_device.hpp"
#include "kf_frame_end.hpp"
#include "kf_icp_grid.hpp"
#include "kf_internal.hpp"
#include "kf_pose_math.hpp"

namespace kf {
namespace {

constexpr int kTerms = 28;   // 21 + 6 + 1 float terms
constexpr int kPad = 32;     // terms padded to a power of two for the wave reduction
constexpr int kSlot = 32;    // doubles per block partial: 28 terms, inliers, candidates, stop marker, unused
constexpr int kInlAt = kTerms, kCandAt = kTerms + 1;
constexpr int kStopAt = kTerms + 2;  // 1 when the block stopped (singular system)
constexpr int kRowPitch = kWave + 4;  // doubles per row entry of a wave's pixels in LDS
constexpr int kThreads = 256;
constexpr double kPivotRelEps = 1e-9;
constexpr int kMinInliers = 6;
constexpr int kFinUnroll = 8;       // slot loads in flight per thread of the slot sum (8 x 32 groups: 256 slots in one round)
// One-block sums and solves use the step's block size, so that every slot sum (in
// a step, the final one-block launch or the single-launch kernel) adds in the same
// order: 32 groups x 16 columns of two doubles of the slots.
constexpr int kSolveThreads = kStepThreads;

struct IcpArgs {
  const float *lvx, *lvy, *lvz, *lnx, *lny, *lnz;  // live level maps (camera frame)
  const float *mvx, *mvy, *mvz, *mnx, *mny, *mnz;  // model level maps (world frame)
  int W, H;
  float fx, fy, cx, cy;
  float dist_thr2;  // sqrtf(d2) < dist_thresh exactly where d2 < dist_thr2
  float cos_thr;
  kf_pose* pose;
  double* partials;
  kf_icp_ctrl* ctrl;
  kf_icp_stats* stats;
  double* sums_out;
  uint8_t* mask;
  int level;
};

// Slot accesses.  COH: relaxed agent-scope atomics, which reach the memory every
// L2 of the chip sees, so blocks can exchange slots across a grid barrier without
// a cache write-back or invalidation (the single-launch form); otherwise ordinary
// accesses, published by a kernel boundary.  The values are the same either way.
template <bool COH>
__device__ __forceinline__ void slot_put(double* p, double v) {
  if constexpr (COH) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *p = v;
}
template <bool COH>
__device__ __forceinline__ double2 slot_get2(const double2* p) {
  if constexpr (COH) {
    double* q = reinterpret_cast<double*>(const_cast<double2*>(p));
    return make_double2(__hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
                        __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  } else {
    return *p;
  }
}

// Association of model pixel i in three phases, so that a thread can issue the
// loads of two pixels before using either: model loads, projection (live pixel
// j), live loads, gating and the row.  Returns 0 = not a candidate, 1 = candidate
// but rejected, 2 = inlier (A, b valid; they are formed for every pixel).
struct PxModel {
  f3 s, m;
  float lz_here;
};
struct PxLive {
  f3 dc, nc;
};

// (byte offsets of a level's pixels fit in 32 bits: sides are at most kMaxImage)
__device__ __forceinline__ PxModel load_model(const IcpArgs& a, int i) {
  const unsigned o = opaque_u32((unsigned)i * 4u);
  return PxModel{f3{plane_at(a.mvx, o), plane_at(a.mvy, o), plane_at(a.mvz, o)},
                 f3{plane_at(a.mnx, o), plane_at(a.mny, o), plane_at(a.mnz, o)}, plane_at(a.lvz, o)};
}

// Live pixel the model point projects to, or -1 (0 = not a candidate, 1 = rejected
// in r when j < 0).  Every value is formed and the tests select the result (a
// wavefront's lanes differ in which test they fail); lanes out of range convert 0.
__device__ __forceinline__ int project_model(const IcpArgs& a, const kf_posef& cw, const PxModel& q, int& r) {
  const bool cand = q.lz_here == q.lz_here && finite3(q.s) && finite3(q.m);
  const f3 sc = xform(cw, q.s);
  const float iz = reciprocal(sc.z);
  const float u = (a.fx * sc.x + a.cx * sc.z) * iz;
  const float v = (a.fy * sc.y + a.cy * sc.z) * iz;
  const float ru = round_half_up(u), rv = round_half_up(v);
  const bool ok = cand && sc.z > 1e-6f && ru >= 0.0f && ru < (float)a.W && rv >= 0.0f && rv < (float)a.H;
  r = cand ? 1 : 0;
  return ok ? (int)(ok ? rv : 0.0f) * a.W + (int)(ok ? ru : 0.0f) : -1;
}

__device__ __forceinline__ PxLive load_live(const IcpArgs& a, int j) {
  const unsigned o = opaque_u32((unsigned)(j < 0 ? 0 : j) * 4u);  // in bounds; unused when j < 0
  return PxLive{f3{plane_at(a.lvx, o), plane_at(a.lvy, o), plane_at(a.lvz, o)},
                f3{plane_at(a.lnx, o), plane_at(a.lny, o), plane_at(a.lnz, o)}};
}

__device__ __forceinline__ int finish_row(const IcpArgs& a, const kf_posef& wc, const PxModel& q, const PxLive& l,
                                          int j, int r, float* A, float& b) {
  // formed for every lane; the gates select the outcome
  const f3 d = xform(wc, l.dc);
  const f3 n = rot(wc.r, l.nc);
  const f3 df = sub(d, q.s);
  const f3 m = q.m, s = q.s;
  const float cs = dot(n, m);
  const bool in = finite3(l.dc) && finite3(l.nc) && dot(df, df) < a.dist_thr2 && cs > a.cos_thr &&
                  cs < 1.0f + 1e-6f;
  A[0] = m.y * d.z - m.z * d.y;
  A[1] = m.z * d.x - m.x * d.z;
  A[2] = m.x * d.y - m.y * d.x;
  A[3] = m.x;
  A[4] = m.y;
  A[5] = m.z;
  b = (m.x * (s.x - d.x) + m.y * (s.y - d.y)) + m.z * (s.z - d.z);
  return j < 0 ? r : (in ? 2 : 1);
}

// Plain mode: adds the 28 terms of one inlier row: 21 upper-triangle A^T A, 6 A^T b, b^2.
__device__ __forceinline__ void accumulate(float* s, const float* A, float b) {
  int k = 0;
#pragma unroll
  for (int p = 0; p < 6; ++p)
#pragma unroll
    for (int q = p; q < 6; ++q) {
      const float v = A[p] * A[q];
      s[k] = s[k] + v;
      ++k;
    }
#pragma unroll
  for (int p = 0; p < 6; ++p) {
    const float v = A[p] * b;
    s[21 + p] = s[21 + p] + v;
  }
  const float v = b * b;
  s[27] = s[27] + v;
}

// One recursive-halving step of the plain mode's wave reduction (reduce-scatter): lanes
// paired by the DPP pattern CTRL hold the same H terms; the lane with `upper` keeps the
// upper H/2, its partner the lower H/2, and each adds the partner's copy of the
// half it keeps.
template <int CTRL, int H>
__device__ __forceinline__ void halve(float* s, bool upper) {
#pragma unroll
  for (int k = 0; k < H / 2; ++k) {
    const float ks = upper ? s[k + H / 2] : s[k];
    const float gs = upper ? s[k] : s[k + H / 2];
    s[k] = ks + dpp_f<CTRL>(gs);
  }
}

// LDS of block_partial.  Compensated mode: the row entries of one round of a wave, one
// pixel per column; the rounds take turns in it (34 KB for eight waves, so that a CU holds
// as many blocks as the registers allow; three rounds' rows side by side, 104 KB, left room
// for one).  Plain mode has no rows.  SETS: sets of wave sums kept at a time.
template <bool COMP, int WAVES, int SETS = 1>
struct PartialLds {
  double rows[COMP ? WAVES : 1][COMP ? 8 : 1][COMP ? kRowPitch : 1];
  double red[SETS][WAVES][kWave];
  int cand[SETS][WAVES];
};

// FP64 sums of products over pixels on v_mfma_f64_4x4x4 (four 4 x 4 products of depth 4
// per instruction, lane l: block b = (l / 4) % 4, operand row l % 4, depth l / 16).  A lane
// reads row entry e = l % 8 of the pixels of its group l / 8 (so 64 lanes hold 8 entries of
// 8 pixels) and the entry 7 - e of the same pixels.  The first register as both operands
// gives the products of entries 0..3 and of entries 4..7 with themselves; the second as
// B the products of 0..3 with 7..4.  Two accumulators each, since a chain waits 24 cycles
// per step.  The LDS reads bound it (eight 16-byte reads per 64 pixels; a lane move in
// place of the second read costs more, operands held per 4 x 4 block twice the reads).
// Against 28 FP64 multiply-adds per thread and a reduce-scatter of 28 doubles over the
// lanes (32 additions, each with four selects and two lane moves): a coarse step's
// association 3.5 k cycles instead of 5.4 k.
struct TermSums {
  double c[2] = {0.0, 0.0}, x[2] = {0.0, 0.0};

  // rows: the wave's 8 x 64 entries in LDS; the pitch puts a quarter-wave's 16-byte
  // reads (8 entries, two pixel pairs) on all 64 banks.
  __device__ __forceinline__ void add(const double (*rows)[kRowPitch]) {
    const int lane = threadIdx.x & 63, e = lane & 7, group = lane >> 3;
    const double2* p = reinterpret_cast<const double2*>(&rows[e][2 * group]);
    const double2* q = reinterpret_cast<const double2*>(&rows[7 - e][2 * group]);
    double2 v[4], w[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {  // pixels 16 u + 2 group, + 1
      v[u] = p[8 * u];
      w[u] = q[8 * u];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      c[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(v[u].x, v[u].x, c[0], 0, 0, 0);
      x[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(v[u].x, w[u].x, x[0], 0, 0, 0);
      c[1] = __builtin_amdgcn_mfma_f64_4x4x4f64(v[u].y, v[u].y, c[1], 0, 0, 0);
      x[1] = __builtin_amdgcn_mfma_f64_4x4x4f64(v[u].y, w[u].y, x[1], 0, 0, 0);
    }
  }
  // The wave's totals: 64 values, see term_of.
  __device__ __forceinline__ void store(double* red) const {
    const int lane = threadIdx.x & 63, at = (lane >> 4) * 8 + (lane & 7);
    const double d = c[0] + c[1], o = x[0] + x[1];
    const double ds = d + dpp_d<0x108>(d), os = o + dpp_d<0x108>(o);  // the two pixel groups of a depth
    if ((lane & 8) == 0) {
      red[at] = ds;
      red[32 + at] = os;
    }
  }
};

// Slot position of the entry (p, q) of R R^T that TermSums leaves at `at`: the term, the
// inlier count (7, 7), or -1 (lower triangles and the other products with the flag).
__device__ __forceinline__ int term_of(int at) {
  const int i = (at >> 3) & 3, b = (at >> 2) & 1, j = at & 3;
  const int p = at < 32 ? 4 * b + i : (b == 0 ? i : 8), q = at < 32 ? 4 * b + j : 7 - j;
  if (p > q) return -1;
  if (q < 6) return p * 6 - p * (p - 1) / 2 + (q - p);
  if (q == 6) return 21 + p;  // A^T b, then b^2 at 27
  return p == 7 ? kInlAt : -1;
}

// Which pixels a block of WAVES waves associates at a time: F full rounds (pixel k nblk T
// + bid T + tid) and, with H, a half round by the block's first WAVES / 2 waves.  nblk
// blocks cover nblk kPixels pixels; larger images repeat.
template <int WAVES, int F, int H>
struct PixelShape {
  static constexpr int T = WAVES * kWave, K = F + H, kPixels = F * T + H * (T / 2);
  __device__ __forceinline__ int pixels() const { return kPixels; }
  // this thread's pixel of round k in pass `pass`; its wave takes part in `rounds` of them
  __device__ __forceinline__ int pixel(int bid, int nblk, int pass, int k) const {
    const int base = pass * nblk * kPixels + k * nblk * T, tid = threadIdx.x;
    return base + (k < F ? bid * T + tid : bid * (T / 2) + tid);
  }
  __device__ __forceinline__ int rounds() const { return H && (int)threadIdx.x >= T / 2 ? F : K; }  // uniform per wave
};

// PixelShape<WAVES, 2, 1> (half) or <WAVES, 3, 0>, chosen at run time: one copy of the code
// in the single-launch kernel, which has little room for registers.
template <int WAVES>
struct WideShape {
  static constexpr int T = WAVES * kWave, K = 3;
  bool half;
  __device__ __forceinline__ int pixels() const { return half ? 2 * T + T / 2 : 3 * T; }
  __device__ __forceinline__ int pixel(int bid, int nblk, int pass, int k) const {
    const int base = pass * nblk * pixels() + k * nblk * T, tid = threadIdx.x;
    return base + (k == 2 && half ? bid * (T / 2) + tid : bid * T + tid);
  }
  __device__ __forceinline__ int rounds() const { return half && (int)threadIdx.x >= T / 2 ? 2 : 3; }
};

// The model samples of a thread's first K pixels in block_partial; they do not
// depend on the pose, so a step can load them before it solves for the pose.
template <int K>
struct PxPre {
  PxModel q[K];
};

template <typename Shape>
__device__ __forceinline__ PxPre<Shape::K> load_models(const IcpArgs& a, const Shape& sh, int bid, int nblk, int pass) {
  const int P = a.W * a.H, rounds = sh.rounds();
  PxPre<Shape::K> pre;
#pragma unroll
  for (int k = 0; k < Shape::K; ++k) {
    const int i = sh.pixel(bid, nblk, pass, k);
    if (k < rounds) pre.q[k] = load_model(a, i < P ? i : 0);  // pixel 0: unused
  }
  return pre;
}

// The sums of one wave over the pixels of its rounds.
template <bool COMP>
struct WaveSums {
  TermSums terms;
  float s[COMP ? 1 : kPad];  // plain mode; terms 28..31 stay zero (padding for the halving)
  int n_in = 0, n_cand = 0;  // of the wave (n_in: plain mode)

  __device__ __forceinline__ WaveSums() {
    if constexpr (!COMP) {
#pragma unroll
      for (int k = 0; k < kPad; ++k) s[k] = 0.0f;
    }
  }

  // The row of a pixel with outcome r (finish_row).  Rejected pixels are zero rows: they
  // leave the sums' bits as they are.  rows: the wave's buffer (compensated mode).
  template <typename Rows>
  __device__ __forceinline__ void add(float* A, float b, int r, Rows& rows) {
    n_cand += (int)__popcll(__ballot(r != 0));
    const bool inl = r == 2;
#pragma unroll
    for (int p = 0; p < 6; ++p) A[p] = inl ? A[p] : 0.0f;
    b = inl ? b : 0.0f;
    if constexpr (COMP) {
      const int lane = threadIdx.x & 63;
      wave_lds_sync();  // the previous round's reads are done
#pragma unroll
      for (int p = 0; p < 6; ++p) rows[p][lane] = (double)A[p];
      rows[6][lane] = (double)b;
      rows[7][lane] = inl ? 1.0 : 0.0;
      wave_lds_sync();
      terms.add(rows);
    } else {
      accumulate(s, A, b);
      n_in += (int)__popcll(__ballot(inl));
    }
  }

  // The wave's totals to red[kWave] and *cand.
  __device__ __forceinline__ void store(double* red, int* cand) {
    const int lane = threadIdx.x & 63;
    if constexpr (COMP) {
      terms.store(red);
    } else {
      // Wave reduction by recursive halving (reduce-scatter): five pairings, each
      // halving the terms a lane holds — row mirror (lane bit 3), half-row mirror
      // (bit 2), quad xor 2 (bit 1), quad xor 1 (bit 0), xor 16 (bit 4) — then xor 32
      // adds the two half-waves.  Lane l < 32 ends with the full wave sum of term
      // 16*b3 + 8*b2 + 4*b1 + 2*b0 + b4 (b = bits of l).
      halve<0x140, 32>(s, (lane & 8) != 0);
      halve<0x141, 16>(s, (lane & 4) != 0);
      halve<0x4E, 8>(s, (lane & 2) != 0);
      halve<0xB1, 4>(s, (lane & 1) != 0);
      const bool up = (lane & 16) != 0;
      const float gs = up ? s[0] : s[1];
      float ks = up ? s[1] : s[0];
      ks = ks + __shfl_xor(gs, 16, kWave);
      ks = ks + __shfl_xor(ks, 32, kWave);
      const int term = ((lane & 8) << 1) | ((lane & 4) << 1) | ((lane & 2) << 1) | ((lane & 1) << 1) | ((lane >> 4) & 1);
      if (lane < 32 && term < kTerms) red[term] = (double)ks;
      if (lane == 32) red[kInlAt] = (double)n_in;
    }
    if (lane == 0) *cand = n_cand;
  }
};

// A slot's terms and inlier count: the sums of its waves' totals, in order (one wave).
template <bool COMP, bool COH>
__device__ __forceinline__ void slot_terms(const double (*red)[kWave], int waves, double* slot) {
  const int lane = threadIdx.x & 63;
  const int at = COMP ? term_of(lane) : (lane <= kInlAt ? lane : -1);
  if (at < 0) return;
  if constexpr (COMP) {
    double S = red[0][lane];
#pragma unroll
    for (int w = 1; w < waves; ++w) S = S + red[w][lane];
    slot_put<COH>(&slot[at], S);
  } else {  // FP32 sums
    float S = (float)red[0][lane];
    for (int w = 1; w < waves; ++w) S = S + (float)red[w][lane];
    slot_put<COH>(&slot[at], (double)S);
  }
}

// Its candidate count and stop marker (one thread).
template <bool COH>
__device__ __forceinline__ void slot_counts(const int* cand, int waves, double* slot) {
  int nc = 0;
  for (int w = 0; w < waves; ++w) nc += cand[w];
  slot_put<COH>(&slot[kCandAt], (double)nc);
  slot_put<COH>(&slot[kStopAt], 0.0);
}

// Block partial: this block's share of the association (K pixels per thread with their
// loads in flight together), the sums over the block's waves, written as one slot: 28
// terms and the inlier and candidate counts.  PRE: the first pass' samples are given.
template <bool COMP, bool PRE = false, bool COH = false, typename Shape, int WAVES, int SETS>
__device__ __forceinline__ void block_partial(const IcpArgs& a, const Shape& sh, const kf_posef& wc, const kf_posef& cw,
                                              int bid, int nblk, double* slot, PartialLds<COMP, WAVES, SETS>& lds,
                                              PxPre<Shape::K> pre = {}) {
  constexpr int K = Shape::K;
  const int tid = threadIdx.x, wave = tid >> 6;
  const int P = a.W * a.H, passes = (P + nblk * sh.pixels() - 1) / (nblk * sh.pixels());
  const int rounds = sh.rounds();
  WaveSums<COMP> sums;
  for (int pass = 0; pass < passes; ++pass) {
    if (!PRE || pass > 0) pre = load_models(a, sh, bid, nblk, pass);
    int j[K], r[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (k >= rounds) continue;  // uniform
      j[k] = project_model(a, cw, pre.q[k], r[k]);
      if (sh.pixel(bid, nblk, pass, k) >= P) {  // no pixel: contributes nothing
        j[k] = -1;
        r[k] = 0;
      }
    }
    PxLive l[K];
#pragma unroll
    for (int k = 0; k < K; ++k)
      if (k < rounds) l[k] = load_live(a, j[k]);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (k >= rounds) continue;
      float A[6], b;
      r[k] = finish_row(a, wc, pre.q[k], l[k], j[k], r[k], A, b);
      const int i = sh.pixel(bid, nblk, pass, k);
      if (a.mask && i < P) a.mask[i] = (uint8_t)(r[k] == 2);
      sums.add(A, b, r[k], lds.rows[COMP ? wave : 0]);
    }
  }
  sums.store(lds.red[0][wave], &lds.cand[0][wave]);
  __syncthreads();
  if (tid < kWave)
    slot_terms<COMP, COH>(lds.red[0], WAVES, slot);
  else if (tid == kWave)
    slot_counts<COH>(lds.cand[0], WAVES, slot);
}

// The partials of several slots by one block, for the shapes of one pixel per thread: a
// round makes one slot or, where a slot has half a block's waves (half), two of them side
// by side; kSlotRounds rounds with their loads in flight together.  Slot i of the block's
// is number first + i * step; those below nb are made, as their own blocks would make them.
constexpr int kSlotRounds = 3;
struct SlotRounds {
  bool half;
  int first, step, nb;
  __device__ __forceinline__ int waves() const { return kStepThreads / kWave >> (int)half; }
  __device__ __forceinline__ int slots() const { return half ? 2 * kSlotRounds : kSlotRounds; }
  __device__ __forceinline__ int number(int i) const { return first + step * i; }
  // this wave's slot in round k, and the thread's pixel of a slot
  __device__ __forceinline__ int slot(int k) const {
    return number(half ? 2 * k + (int)(threadIdx.x / (kStepThreads / 2)) : k);
  }
  __device__ __forceinline__ int pixel(int v) const {
    return half ? v * (kStepThreads / 2) + (int)threadIdx.x % (kStepThreads / 2) : v * kStepThreads + (int)threadIdx.x;
  }
};

__device__ __forceinline__ PxPre<kSlotRounds> load_slot_models(const IcpArgs& a, const SlotRounds& sr) {
  const int P = a.W * a.H;
  PxPre<kSlotRounds> pre;
#pragma unroll
  for (int k = 0; k < kSlotRounds; ++k) {
    const int v = sr.slot(k), i = sr.pixel(v);
    if (v < sr.nb) pre.q[k] = load_model(a, i < P ? i : 0);  // uniform per wave; pixel 0: unused
  }
  return pre;
}

template <bool COMP, int WAVES>
__device__ __forceinline__ void slot_partials(const IcpArgs& a, const SlotRounds& sr, const kf_posef& wc, const kf_posef& cw,
                                              double* slots, PartialLds<COMP, WAVES, kSlotRounds>& lds,
                                              const PxPre<kSlotRounds>& pre) {
  static_assert(WAVES * kWave == kStepThreads && 2 * kSlotRounds <= WAVES, "a wave per slot at the end");
  const int wave = threadIdx.x >> 6, P = a.W * a.H;
  int j[kSlotRounds], r[kSlotRounds];
#pragma unroll
  for (int k = 0; k < kSlotRounds; ++k) {
    const int v = sr.slot(k);
    if (v >= sr.nb) continue;  // uniform per wave
    j[k] = project_model(a, cw, pre.q[k], r[k]);
    if (sr.pixel(v) >= P) {
      j[k] = -1;
      r[k] = 0;
    }
  }
  PxLive l[kSlotRounds];
#pragma unroll
  for (int k = 0; k < kSlotRounds; ++k)
    if (sr.slot(k) < sr.nb) l[k] = load_live(a, j[k]);
#pragma unroll
  for (int k = 0; k < kSlotRounds; ++k) {
    if (sr.slot(k) >= sr.nb) continue;
    float A[6], b;
    r[k] = finish_row(a, wc, pre.q[k], l[k], j[k], r[k], A, b);
    WaveSums<COMP> sums;
    sums.add(A, b, r[k], lds.rows[COMP ? wave : 0]);
    sums.store(lds.red[k][wave], &lds.cand[k][wave]);
  }
  __syncthreads();
  if (wave < sr.slots() && sr.number(wave) < sr.nb) {
    const int k = sr.half ? wave / 2 : wave, w0 = sr.half ? wave % 2 * (WAVES / 2) : 0;
    double* slot = slots + (size_t)sr.number(wave) * kSlot;
    slot_terms<COMP, true>(lds.red[k] + w0, sr.waves(), slot);
    if ((threadIdx.x & 63) == 0) slot_counts<true>(lds.cand[k] + w0, sr.waves(), slot);
  }
}

// x of the lane 16 (32) away added to this lane's (v_permlane16_swap / 32_swap: the two
// results are the lower and the upper rows' values in every lane).
__device__ __forceinline__ double add_rows16(double x) {
  const uint2 u = __builtin_bit_cast(uint2, x);
  const auto lo = __builtin_amdgcn_permlane16_swap(u.x, u.x, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(u.y, u.y, false, false);
  return __builtin_bit_cast(double, make_uint2(lo[0], hi[0])) + __builtin_bit_cast(double, make_uint2(lo[1], hi[1]));
}
__device__ __forceinline__ double add_rows32(double x) {
  const uint2 u = __builtin_bit_cast(uint2, x);
  const auto lo = __builtin_amdgcn_permlane32_swap(u.x, u.x, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(u.y, u.y, false, false);
  return __builtin_bit_cast(double, make_uint2(lo[0], hi[0])) + __builtin_bit_cast(double, make_uint2(lo[1], hi[1]));
}

// FP64 sum of nb slots: thread (g, j) reads doubles 2j, 2j + 1 of slots g, g + G, ...
// with kFinUnroll loads in flight; the groups of a wave are added by lane moves and
// each wave leaves its 32 sums in fin[wave] (publish with a barrier, then
// wave_totals).  Split in two so that a caller can issue the first round of slot loads
// before other loads (loads complete in issue order) and consume them later.  COH: the
// slots were written across a grid barrier.
template <int THREADS>
struct SlotFin {
  double w[THREADS / kWave][kSlot];
};

template <int THREADS, bool COH = false>
struct SlotSum {
  static constexpr int G = THREADS / 16;
  double2 v[kFinUnroll];
  // The first round of loads (slots g, g + G, ..., g + (kFinUnroll - 1) G; nb >= 1).
  // Unconditional, from clamped in-bounds addresses, so that nothing waits for
  // them here; reduce() drops the out-of-range ones.
  __device__ __forceinline__ void load(const double* slots, int nb) {
    const int j = threadIdx.x & 15, g = threadIdx.x >> 4;
    const double2* base = reinterpret_cast<const double2*>(slots) + j;
#pragma unroll
    for (int u = 0; u < kFinUnroll; ++u) v[u] = slot_get2<COH>(base + (size_t)min(g + G * u, nb - 1) * (kSlot / 2));
  }
  __device__ __forceinline__ void reduce(const double* slots, int nb, SlotFin<THREADS>& fin) {
    const int tid = threadIdx.x, j = tid & 15, g = tid >> 4;
    const double2* base = reinterpret_cast<const double2*>(slots) + j;
    double a0 = 0.0, a1 = 0.0;
    for (int b0 = g;;) {
#pragma unroll
      for (int u = 0; u < kFinUnroll; ++u) {
        const bool in = b0 + G * u < nb;
        a0 = a0 + (in ? v[u].x : 0.0);
        a1 = a1 + (in ? v[u].y : 0.0);
      }
      b0 += G * kFinUnroll;
      if (b0 - g >= nb) break;  // uniform
#pragma unroll
      for (int u = 0; u < kFinUnroll; ++u) v[u] = slot_get2<COH>(base + (size_t)min(b0 + G * u, nb - 1) * (kSlot / 2));
    }
    a0 = add_rows32(add_rows16(a0));
    a1 = add_rows32(add_rows16(a1));
    if ((tid & 63) < 16) {
      fin.w[tid >> 6][2 * j] = a0;
      fin.w[tid >> 6][2 * j + 1] = a1;
    }
  }
};

// Slot sum lane % 32, from the waves' sums in order (any wave, after the barrier).
template <int THREADS>
__device__ __forceinline__ double wave_totals(const SlotFin<THREADS>& fin) {
  const int t = threadIdx.x & (kSlot - 1);
  double s = fin.w[0][t];
#pragma unroll
  for (int w = 1; w < THREADS / kWave; ++w) s = s + fin.w[w][t];
  return s;
}

// Lane l's value of v, in every lane (v_readlane: no LDS round trip).
__device__ __forceinline__ double lane_value(double v, int l) {
  const long long b = __builtin_bit_cast(long long, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(b & 0xffffffffll), l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), l);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// Solve (A^T A) x = A^T b from the slot sums in fin (published) and compose the
// Euler-ZYX increment onto Tin (LDS, 16 doubles): Tout (LDS) and the FP32 fields
// wc / cw (LDS).  Returns false, with the outputs untouched, when an earlier solve was
// singular (a block stopped) or this one is (fewer than kMinInliers inliers or an
// LDL^T pivot not above 1e-9 x the largest diagonal).  With `st`, the level statistics
// are written and, when this system is singular, status 1.
// Called by the whole block; the first wavefront computes, as one chain of dependent
// FP64 operations: every lane solves with the square-root-free factorisation shared with
// the host (ldlt_solve6: no branch, and no broadcast of the solution after it), lanes
// 0..2 take the sine and cosine of one angle each (v_readlane), lane 4i + j forms entry
// (i, j) of the product with the expressions of the serial helpers, and the FP32
// field(s) that entry gives; the rigid inverse's translation sums down the columns by
// DPP row shifts.  The statistics (a division and a square root) are written by the
// second wavefront meanwhile; the final barrier publishes everything.  3.1 k cycles from
// the slot sums to the barrier against 4.1 k with lane 0 alone in the factorisation, IEEE
// divisions and 24 lane broadcasts for the inverse.
template <int THREADS>
__device__ __forceinline__ bool solve_compose(const SlotFin<THREADS>& fin, const double* Tin, kf_icp_stats* st, int level,
                                              double* Tout, kf_posef* wc, kf_posef* cw) {
  __shared__ int tok;
  __shared__ __align__(16) double sum[kSlot];
  const int tid = threadIdx.x;
  if (tid < kWave) {
    const int lane = tid;
    const int i = (lane >> 2) & 3, j = lane & 3;
    // this lane's column of Tin (for the product), loaded before the solve
    const double b0 = Tin[j], b1 = Tin[4 + j], b2 = Tin[8 + j], b3 = Tin[12 + j];
    const double tot = wave_totals(fin);
    if (lane < kSlot) sum[lane] = tot;
    wave_lds_sync();
    double up[21], g[6], x[6];
#pragma unroll
    for (int q = 0; q < 21; ++q) up[q] = sum[q];
#pragma unroll
    for (int q = 0; q < 6; ++q) g[q] = sum[21 + q];
    const bool stopped = sum[kStopAt] != 0.0, few = (int)sum[kInlAt] < kMinInliers;
    const bool solved = ldlt_solve6(up, g, kPivotRelEps, x) && !few;
    const int ok = __builtin_amdgcn_readfirstlane(!stopped && solved ? 1 : 0);  // every lane agrees
    if (lane == 0) {
      tok = ok;
      if (!stopped && !ok && st) st->status = 1;
    }
    if (ok) {  // uniform
      // lanes 0, 1, 2: the angle of their axis (the rotation is the negated solution)
      const double ang = -(lane == 0 ? x[0] : (lane == 1 ? x[1] : x[2]));
      double cl, sl;
      small_sincos(ang, &cl, &sl);
      const double c0 = lane_value(cl, 0), s0 = lane_value(sl, 0);
      const double c1 = lane_value(cl, 1), s1 = lane_value(sl, 1);
      const double c2 = lane_value(cl, 2), s2 = lane_value(sl, 2);
      double D[12];
#pragma unroll
      for (int e = 0; e < 12; ++e) D[e] = euler_zyx_entry(e, c0, s0, c1, s1, c2, s2, x[3], x[4], x[5]);
      // row i of the increment (rows 0..2; row 3 is (0, 0, 0, 1))
      const double a0 = i == 0 ? D[0] : (i == 1 ? D[4] : D[8]);
      const double a1 = i == 0 ? D[1] : (i == 1 ? D[5] : D[9]);
      const double a2 = i == 0 ? D[2] : (i == 1 ? D[6] : D[10]);
      const double a3 = i == 0 ? D[3] : (i == 1 ? D[7] : D[11]);
      // entry (i, j) of D * Tin in mat4_mul_entry's order
      const double t = (i == 3) ? (j == 3 ? 1.0 : 0.0) : ((a0 * b0 + a1 * b1) + a2 * b2) + a3 * b3;
      if (lane < 16) Tout[lane] = t;
      if (lane < 12) {
        const float f = (float)t;
        if (j < 3) {
          wc->r[i * 3 + j] = f;
          cw->r[j * 3 + i] = f;  // cw = rigid inverse: R^T and -R^T t
        } else {
          wc->t[i] = f;
        }
      }
      // -(R^T t), rows 0..2 in rigid_inverse_t's order: R(i, c) t_i, t_i from the quad's
      // last lane, then rows 1 and 2 of the column from 4 and 8 lanes up
      const double p = t * dpp_d<0xFF>(t);
      const double r = (p + dpp_d<0x104>(p)) + dpp_d<0x108>(p);
      if (lane < 3) cw->t[lane] = (float)-r;
    }
  } else if (tid < 2 * kWave && st) {
    const double tot = wave_totals(fin);
    const double b2 = lane_value(tot, 27), inl = lane_value(tot, kInlAt), cand = lane_value(tot, kCandAt);
    if (tid == kWave && lane_value(tot, kStopAt) == 0.0) {
      const int ni = (int)inl;
      const double rms = ni > 0 ? sqrt(b2 / inl) : 0.0;
      st->inliers = ni;
      st->candidates = (int)cand;
      st->residual_rms = rms;
      st->level_residual[level] = rms;
      st->level_inliers[level] = ni;
    }
  }
  __syncthreads();
  return tok != 0;  // uniform
}

// Copies a pose (thread-parallel, 28 words of 8 bytes).
__device__ __forceinline__ void copy_pose(const kf_pose* src, kf_pose* dst) {
  static_assert(sizeof(kf_pose) % 8 == 0, "pose size");
  const int n = (int)(sizeof(kf_pose) / 8);
  if ((int)threadIdx.x < n)
    reinterpret_cast<unsigned long long*>(dst)[threadIdx.x] = reinterpret_cast<const unsigned long long*>(src)[threadIdx.x];
}

// Reduce mode (kf_icp_reduce), pass 1: the block partials at a fixed pose.
template <bool COMP>
__global__ __launch_bounds__(kThreads) void icp_partials(IcpArgs a) {
  const PixelShape<kThreads / kWave, 2, 0> shape;
  __shared__ PartialLds<COMP, kThreads / kWave> lds;
  const kf_posef wc = a.pose->wc, cw = a.pose->cw;
  block_partial<COMP>(a, shape, wc, cw, blockIdx.x, gridDim.x, a.partials + (size_t)blockIdx.x * kSlot, lds);
}

// Reduce mode, pass 2 (one block): the FP64 sums.
__global__ __launch_bounds__(kSolveThreads) void icp_sums(IcpArgs a, int nb) {
  __shared__ SlotFin<kSolveThreads> fin;
  SlotSum<kSolveThreads> slots;
  slots.load(a.partials, nb);
  slots.reduce(a.partials, nb, fin);
  __syncthreads();
  const double tot = wave_totals(fin);
  if ((int)threadIdx.x < kTerms + 2) a.sums_out[threadIdx.x] = tot;
}

// Tracking: one launch per iteration.  Every block first solves the previous
// iteration from its slots (the same FP64 sums, solve and composition in every
// block, so all blocks agree bit for bit on the new pose; block 0 publishes it
// and the statistics), then associates with the new pose and writes its slot.
// Poses and slots alternate between two buffers, so no block overwrites what
// another block of the same launch still reads; a kernel boundary publishes
// them (one launch per iteration instead of a partials and a solve launch).
struct StepArgs {
  const kf_pose* pose_in;   // the guess (first step) or the previous step's output
  kf_pose* pose_out;
  const double* slots_in;   // previous step's slots (unused for the first step)
  double* slots_out;
  int nb_in;                // number of slots in slots_in
  int level_in;             // level of the previous step
  int first;
  int index;                 // step number in the call (step k solves iteration k - 1)
  const kf_icp_stats* user;  // its skip flag makes icp_finish leave the outputs untouched
                             // (the tracker's own statistics when the caller passes none)
  kf_icp_stats* st;
};

// F, H: the pixels a thread takes at this level's grid (PixelShape; the model samples of
// all of them are loaded before the solve).
template <int F, int H>
using StepShape = PixelShape<kStepThreads / kWave, F, H>;

template <bool COMP, int F, int H>
__global__ __launch_bounds__(kStepThreads) void icp_step(IcpArgs a, StepArgs S) {
  __shared__ double Tin[16], Tnew[16];
  __shared__ kf_posef s_wc, s_cw;
  __shared__ SlotFin<kStepThreads> fin;
  const StepShape<F, H> shape;
  __shared__ PartialLds<COMP, kStepThreads / kWave> lds;
  const int tid = threadIdx.x;
  double* slot_out = S.slots_out + (size_t)blockIdx.x * kSlot;
  // Every load that does not depend on another is issued up front, in the order
  // they are needed (loads complete in issue order): the previous step's slots
  // and pose, then the model samples.  No flag is read before them: a singular
  // solve is passed on through the slots' stop markers.
  SlotSum<kStepThreads> slots_in;
  double tin = 0.0;
  if (!S.first) {
    slots_in.load(S.slots_in, S.nb_in);
    tin = S.pose_in->T_wc[tid & 15];
  }
  const PxPre<F + H> pre = load_models(a, shape, blockIdx.x, gridDim.x, 0);
  if (S.first) {
    if (tid < 12) {
      if (tid < 9) s_wc.r[tid] = S.pose_in->wc.r[tid];
      else s_wc.t[tid - 9] = S.pose_in->wc.t[tid - 9];
    } else if (tid < 24) {
      if (tid < 21) s_cw.r[tid - 12] = S.pose_in->cw.r[tid - 12];
      else s_cw.t[tid - 21] = S.pose_in->cw.t[tid - 21];
    }
    if (blockIdx.x == 0) {
      copy_pose(S.pose_in, S.pose_out);
      if (tid == 32) {
        a.ctrl->executed = 0;
        kf_icp_stats z = {};
        *S.st = z;
      }
    }
  } else {
    slots_in.reduce(S.slots_in, S.nb_in, fin);
    if (tid < 16) Tin[tid] = tin;
    __syncthreads();
    // an earlier solve was singular (a previous block stopped), or this one is:
    // keep the pose and pass the stop on
    if (!solve_compose(fin, Tin, blockIdx.x == 0 ? S.st : nullptr, S.level_in, Tnew, &s_wc, &s_cw)) {
      if (blockIdx.x == 0) copy_pose(S.pose_in, S.pose_out);
      if (tid == 0) slot_out[kStopAt] = 1.0;
      return;  // uniform
    }
    if (blockIdx.x == 0) {
      kf_pose* P = S.pose_out;
      if (tid < 16) P->T_wc[tid] = Tnew[tid];
      else if (tid >= 64 && tid < 76) {
        const int q = tid - 64;
        if (q < 9) P->wc.r[q] = s_wc.r[q]; else P->wc.t[q - 9] = s_wc.t[q - 9];
      } else if (tid >= 128 && tid < 140) {
        const int q = tid - 128;
        if (q < 9) P->cw.r[q] = s_cw.r[q]; else P->cw.t[q - 9] = s_cw.t[q - 9];
      } else if (tid == 192) {
        a.ctrl->executed = S.index;  // every earlier solve succeeded too
      }
    }
  }
  __syncthreads();
  block_partial<COMP, true>(a, shape, s_wc, s_cw, blockIdx.x, gridDim.x, slot_out, lds, pre);
}

// Acceptance test of the finished call (IcpGate), from the window count and thread
// i's window entry (wv = window[i] for i < window_len), loaded by the caller at its
// start.  The window's median: lane i ranks value i (ties broken by index) and the
// lanes of the middle rank(s) publish their values, one pass instead of a serial
// sort.  Every thread of the block calls it.
__device__ void gate_decide(const IcpGate& g, int count, double wv, const kf_icp_stats* sp, const kf_pose* pose) {
  __shared__ double v[kGateMaxWindow], mid[2];
  __shared__ int s_fail;
  const int i = threadIdx.x;
  const int n = min(count, g.window_len);
  if (i < n) v[i] = wv;
  __syncthreads();
  if (i < n) {
    const double x = v[i];
    int rank = 0;
    for (int j = 0; j < n; ++j) rank += (v[j] < x || (v[j] == x && j < i)) ? 1 : 0;
    if (rank == n / 2) mid[1] = x;
    if ((n & 1) == 0 && rank == n / 2 - 1) mid[0] = x;
  }
  __syncthreads();
  if (i == 0) {
    bool fail = sp->status != 0 || sp->iterations == 0 || !(sp->residual_rms == sp->residual_rms);
    if (!fail && sp->candidates > 0 && (double)sp->inliers < (double)g.min_frac * (double)sp->candidates)
      fail = true;
    if (!fail && n >= g.window_min) {
      const double med = (n & 1) ? mid[1] : 0.5 * (mid[0] + mid[1]);
      if (sp->residual_rms > (double)g.ratio * med) fail = true;
    }
    *g.used = 1;
    *g.fell_back = fail ? 1 : 0;
    g.fallback->skip = fail ? 0 : 1;
    s_fail = fail ? 1 : 0;
  }
  __syncthreads();
  if (!s_fail) copy_pose(pose, g.accept_out);
}

// End of tracking (one block): solves the last step's slots, writes the output
// pose and the statistics (iterations = updates applied), copies them to the
// caller's statistics, then runs the acceptance test when gated.  `steps` = 0: no
// step ran; the guess is the result.
__global__ __launch_bounds__(kSolveThreads) void icp_finish(IcpArgs a, StepArgs S, int steps, kf_pose* out,
                                                            kf_icp_stats* user, IcpGate gate, int gated,
                                                            FrameEnd fe, int fe_on) {
  __shared__ double Tin[16];
  __shared__ SlotFin<kSolveThreads> fin;
  // The call's statistics and output pose are assembled in LDS and stored once; the
  // acceptance test reads them there instead of back from memory.
  __shared__ kf_icp_stats s_st;
  __shared__ kf_pose s_out;
  constexpr int kStWords = (int)(sizeof(kf_icp_stats) / 8), kPoseWords = (int)(sizeof(kf_pose) / 8);
  static_assert(sizeof(kf_icp_stats) % 8 == 0 && sizeof(kf_pose) % 8 == 0, "8-byte words");
  const int tid = threadIdx.x;
  // Every independent load first (loads complete in issue order): the skip flag, the
  // last step's slots and pose, the statistics and the count of applied updates so
  // far, the acceptance test's window.  A skipped call (uniform) computes like any
  // other into the tracker's own statistics and leaves the caller's pose and
  // statistics untouched.
  const int skip = S.user->skip;
  SlotSum<kSolveThreads> slots_in;
  double tin = 0.0;
  if (steps > 0) {
    slots_in.load(S.slots_in, S.nb_in);
    tin = S.pose_in->T_wc[tid & 15];
  }
  unsigned long long stw = 0ull, pw = 0ull;
  if (tid < kStWords) stw = reinterpret_cast<const unsigned long long*>(S.st)[tid];
  if (tid >= kWave && tid < kWave + kPoseWords) pw = reinterpret_cast<const unsigned long long*>(S.pose_in)[tid - kWave];
  const int exec_prev = tid == 0 ? a.ctrl->executed : 0;
  int gcount = 0;
  double gwv = 0.0;
  if (gated) {
    gcount = *gate.count;
    gwv = gate.window[min(tid, gate.window_len - 1)];
  }
  // the statistics start from their stored state (all zero when no step ran) and
  // the output pose from the input one (kept when no update applies)
  if (tid < kStWords) reinterpret_cast<unsigned long long*>(&s_st)[tid] = steps > 0 ? stw : 0ull;
  if (tid >= kWave && tid < kWave + kPoseWords) reinterpret_cast<unsigned long long*>(&s_out)[tid - kWave] = pw;
  bool ok = false;
  if (steps == 0) {
    if (tid == 32) a.ctrl->executed = 0;
    __syncthreads();
  } else {
    slots_in.reduce(S.slots_in, S.nb_in, fin);
    if (tid < 16) Tin[tid] = tin;
    __syncthreads();  // also publishes s_st and s_out
    ok = solve_compose(fin, Tin, &s_st, S.level_in, s_out.T_wc, &s_out.wc, &s_out.cw);
    if (ok && tid == 192) a.ctrl->executed = steps;
  }
  // iterations = updates applied: every step's when the last solve succeeded, else
  // those counted by the steps
  if (tid == 0) s_st.iterations = steps == 0 ? 0 : (ok ? steps : exec_prev);
  __syncthreads();
  if (tid < kStWords) reinterpret_cast<unsigned long long*>(S.st)[tid] = reinterpret_cast<const unsigned long long*>(&s_st)[tid];
  if (!skip) {  // uniform
    if (user && user != S.st && tid >= 32 && tid < 32 + kStWords) {
      constexpr int so = (int)offsetof(kf_icp_stats, skip);
      unsigned long long w = reinterpret_cast<const unsigned long long*>(&s_st)[tid - 32];
      if (tid - 32 == so / 8) w &= ~(0xffffffffull << (8 * (so % 8)));  // the caller's copy: skip = 0
      reinterpret_cast<unsigned long long*>(user)[tid - 32] = w;
    }
    if (tid >= kWave && tid < kWave + kPoseWords)
      reinterpret_cast<unsigned long long*>(out)[tid - kWave] = reinterpret_cast<const unsigned long long*>(&s_out)[tid - kWave];
  }
  if (gated && !skip) {  // uniform
    __syncthreads();
    gate_decide(gate, gcount, gwv, &s_st, &s_out);
  }
  if (fe_on) {  // uniform
    __syncthreads();
    frame_end_run(fe);
  }
}

// ---------------------------------------------------------------------------
// Single-launch tracking: the iterations of the icp_step chain and icp_finish in
// one launch.  Block b computes the slots b, b + G, ... of each iteration's step
// grid (the same pixels and sums per slot, hence the same slots), every block sums the previous iteration's slots and solves as
// icp_step does, and a grid barrier replaces the kernel boundary between
// iterations, so poses and statistics are those of the multi-launch chain bit for
// bit.  Every block keeps the pose in LDS; only the lead block writes it, then runs
// the acceptance test (when gated) and the frame-end bookkeeping, as icp_finish.
//
// The barrier needs all G blocks resident at once: the launcher caps G at the
// device's co-resident block count for this kernel, and keeps it well below where
// several calls of one size fit together (chain_blocks).  Its wait is bounded: a block
// that waits longer than the control block's poll limit (kBarrierPolls unless set
// with kf_tracker_set_barrier_polls) gives up, the control block is marked
// broken and that call and every later single-launch call of the tracker report
// status 2 until kf_tracker_reset (the waits of the other blocks end the same
// way), so the grid always drains.
constexpr unsigned kBarrierPolls = 1u << 20;

struct ChainArgs {
  IcpArgs lv[KF_MAX_LEVELS];
  int levels;
  int iters[KF_MAX_LEVELS];
  int blocks[KF_MAX_LEVELS];  // step grid (slot count) per level, as in the multi-launch chain
  int shape[KF_MAX_LEVELS];   // pixels per thread of that grid (step_shape), as in the multi-launch chain
  const kf_pose* guess;
  kf_pose* out;
  double* slots[2];
  kf_icp_stats* user;  // skip flag; receives a copy of the statistics
  kf_icp_stats* st;
  kf_icp_ctrl* ctrl;
  IcpGate gate;        // evaluated by the lead block at the end when gated
  int gated;
  FrameEnd fe;         // run by the lead block at the end when fe_on
  int fe_on;
};

__device__ __forceinline__ unsigned ctrl_load(const unsigned* p) {
  return __hip_atomic_load(const_cast<unsigned*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void ctrl_store(unsigned* p, unsigned v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned ctrl_add(unsigned* p) {
  return __hip_atomic_fetch_add(p, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Grid barrier, two levels: block b arrives on the counter of group b mod 8; the
// last arrival of a group arrives on the top counter; the last of those has seen
// every block arrive, so it clears the counters (nothing touches them again before
// the release) and releases the grid by storing the barrier's number into the
// generation word that the others poll.  Each counter sits on a line of its own,
// so at most ceil(G / 8) + 8 atomics queue on one address instead of G.  All
// accesses are relaxed agent-scope atomics (no cache write-back): the slots they
// publish are written and read with the same kind of access, and every store a
// block issued has completed (s_waitcnt 0, which counts stores on this chip) before
// its arrival; a released block reads the slots only after it saw the release.
// `target`: this barrier's generation (thread 0's; the previous one + 1).
// Returns false (for the whole block) when the wait timed out.
__device__ __forceinline__ bool grid_barrier(kf_icp_ctrl* ctrl, unsigned target, unsigned limit) {
  __shared__ int s_ok;
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0) {
    int ok = 1;
    const unsigned G = gridDim.x, g = blockIdx.x & 7;
    const unsigned members = (G - g + 7) / 8, groups = G < 8 ? G : 8;
    bool last = ctrl_add(&ctrl->group[g][0]) == members - 1;
    if (last) last = ctrl_add(&ctrl->top) == groups - 1;
    if (last) {
      for (unsigned q = 0; q < groups; ++q) ctrl_store(&ctrl->group[q][0], 0u);
      ctrl_store(&ctrl->top, 0u);
      __builtin_amdgcn_s_waitcnt(0);  // the counters are clear before anyone is released
      ctrl_store(&ctrl->gen, target);
    } else {
      unsigned polls = 0;
      while ((int)(ctrl_load(&ctrl->gen) - target) < 0) {
        if (++polls >= limit) {
          ok = 0;
          __hip_atomic_store(&ctrl->broken, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
    }
    s_ok = ok;
  }
  __syncthreads();
  return s_ok != 0;
}

// One iteration of the chain at a level whose step grid has nb blocks of the given shape
// (as icp_step): the slot loads of the previous iteration
// (solve = true; nb_in slots of level lvl_in), then this block's model samples, both
// in flight together; the sum, solve and composition onto T[cur]; this block's slots,
// several at once in the shapes of one pixel per thread (WIDE = false).  half: the shape
// ends in half a block's pixels.  Returns false (uniform) when the solve was singular:
// nothing is written.
template <bool COMP, bool WIDE, typename Lds>
__device__ __forceinline__ bool chain_iteration(const IcpArgs& a, bool half, int nb, bool solve, const double* slots_in,
                                                int nb_in, int lvl_in, double* slots_out,
                                                SlotFin<kStepThreads>& fin, Lds& lds,
                                                double (*T)[16], int& cur, kf_posef* wc, kf_posef* cw,
                                                kf_icp_stats* st) {
  const WideShape<kStepThreads / kWave> shape{half};
  SlotRounds sr{half, (int)blockIdx.x, (int)gridDim.x, nb};
  SlotSum<kStepThreads, true> L;
  if (solve) L.load(slots_in, nb_in);
  PxPre<3> pre = {};
  auto load = [&]() {
    if constexpr (WIDE)
      pre = load_models(a, shape, sr.first, nb, 0);
    else
      pre = load_slot_models(a, sr);
  };
  if (sr.first < nb) load();
  if (solve) {
    L.reduce(slots_in, nb_in, fin);
    __syncthreads();
    if (!solve_compose(fin, T[cur], st, lvl_in, T[cur ^ 1], wc, cw)) return false;
    cur ^= 1;
  }
  __syncthreads();
  while (sr.first < nb) {  // uniform
    if constexpr (WIDE)
      block_partial<COMP, true, true>(a, shape, *wc, *cw, sr.first, nb, slots_out + (size_t)sr.first * kSlot, lds, pre);
    else
      slot_partials<COMP>(a, sr, *wc, *cw, slots_out, lds, pre);
    sr.first += sr.step * (WIDE ? 1 : sr.slots());
    if (sr.first < nb) {
      load();
      __syncthreads();
    }
  }
  return true;
}

template <bool COMP>
__global__ __launch_bounds__(kStepThreads) void icp_chain(ChainArgs C) {
  __shared__ double T[2][16];
  __shared__ kf_posef s_wc, s_cw;
  __shared__ SlotFin<kStepThreads> fin;
  __shared__ PartialLds<COMP, kStepThreads / kWave, kSlotRounds> lds;
  const int tid = threadIdx.x;
  const bool lead = blockIdx.x == 0;
  if (C.user && C.user->skip) {  // uniform
    if (lead && C.fe_on) frame_end_run(C.fe);
    return;
  }
  kf_icp_stats* st = C.st;
  if (C.ctrl->broken) {  // uniform: written by an earlier launch
    if (lead && tid == 0) {
      kf_icp_stats z = {};
      z.status = 2;
      *st = z;
      if (C.user && C.user != st) *C.user = z;
    }
    if (lead) copy_pose(C.guess, C.out);
    if (lead && C.gated) {
      __syncthreads();
      gate_decide(C.gate, *C.gate.count, C.gate.window[min(tid, C.gate.window_len - 1)], st, C.out);
    }
    if (lead && C.fe_on) {
      __syncthreads();
      frame_end_run(C.fe);
    }
    return;
  }
  // barrier state (thread 0): the generation before this launch's first barrier
  // (it cannot advance before this block arrives there) and the poll bound
  unsigned gen = 0, limit = kBarrierPolls;
  if (tid == 0) {
    gen = ctrl_load(&C.ctrl->gen);
    const unsigned pl = C.ctrl->poll_limit;
    limit = pl ? pl : kBarrierPolls;
  }
  int gcount = 0;
  double gwv = 0.0;
  if (lead && C.gated) {
    gcount = *C.gate.count;
    gwv = C.gate.window[min(tid, C.gate.window_len - 1)];
  }
  if (tid < 16) T[0][tid] = C.guess->T_wc[tid];
  if (tid < 12) {
    if (tid < 9) s_wc.r[tid] = C.guess->wc.r[tid];
    else s_wc.t[tid - 9] = C.guess->wc.t[tid - 9];
  } else if (tid < 24) {
    if (tid < 21) s_cw.r[tid - 12] = C.guess->cw.r[tid - 12];
    else s_cw.t[tid - 21] = C.guess->cw.t[tid - 21];
  }
  if (lead && tid == 32) {
    kf_icp_stats z = {};
    *st = z;
  }
  __syncthreads();
  int cur = 0, executed = 0, nb_prev = 0, lvl_prev = 0, par = 0, steps = 0;
  bool stop = false, timeout = false;
  for (int l = C.levels - 1; l >= 0 && !stop; --l) {
    const IcpArgs& a = C.lv[l];
    const int nb = C.blocks[l];
    for (int it = 0; it < C.iters[l]; ++it) {
      const bool solve = steps > 0;
      kf_icp_stats* sp = lead ? st : nullptr;
      const int shape = C.shape[l];  // uniform
      const bool half = shape == 0 || shape == 2;
      const bool ok = shape < 2 ? chain_iteration<COMP, false>(a, half, nb, solve, C.slots[par ^ 1], nb_prev, lvl_prev,
                                                               C.slots[par], fin, lds, T, cur, &s_wc, &s_cw, sp)
                                : chain_iteration<COMP, true>(a, half, nb, solve, C.slots[par ^ 1], nb_prev, lvl_prev,
                                                              C.slots[par], fin, lds, T, cur, &s_wc, &s_cw, sp);
      if (!ok) {
        stop = true;  // uniform: every block solved the same system
        break;
      }
      if (solve) ++executed;
      if (!grid_barrier(C.ctrl, ++gen, limit)) {
        stop = timeout = true;
        break;
      }
      nb_prev = nb;
      lvl_prev = l;
      par ^= 1;
      ++steps;
    }
  }
  if (!stop && steps > 0) {  // the last iteration's update (as icp_finish)
    SlotSum<kStepThreads, true> L;
    L.load(C.slots[par ^ 1], nb_prev);
    L.reduce(C.slots[par ^ 1], nb_prev, fin);
    __syncthreads();
    if (solve_compose(fin, T[cur], lead ? st : nullptr, lvl_prev, T[cur ^ 1], &s_wc, &s_cw)) {
      cur ^= 1;
      ++executed;
    }
  }
  if (!lead) return;
  __syncthreads();
  kf_pose* P = C.out;
  if (tid < 16) P->T_wc[tid] = T[cur][tid];
  else if (tid >= 64 && tid < 76) {
    const int q = tid - 64;
    if (q < 9) P->wc.r[q] = s_wc.r[q]; else P->wc.t[q - 9] = s_wc.t[q - 9];
  } else if (tid >= 128 && tid < 140) {
    const int q = tid - 128;
    if (q < 9) P->cw.r[q] = s_cw.r[q]; else P->cw.t[q - 9] = s_cw.t[q - 9];
  }
  __syncthreads();
  if (tid == 0) {
    st->iterations = executed;
    if (timeout) st->status = 2;
    if (C.user && C.user != st) {
      kf_icp_stats c = *st;
      c.skip = 0;
      *C.user = c;
    }
  }
  if (C.gated) {
    __syncthreads();
    gate_decide(C.gate, gcount, gwv, st, C.out);
  }
  if (C.fe_on) {
    __syncthreads();
    frame_end_run(C.fe);
  }
}

__global__ void pose_const_velocity(const kf_pose* p2, const kf_pose* p1, kf_pose* g) {
  if (threadIdx.x != 0) return;
  *g = constant_velocity_pose(*p2, *p1);
}

__global__ void pose_copy(const kf_pose* src, kf_pose* dst) {
  if (threadIdx.x == 0) *dst = *src;
}

// The smallest float whose square root (correctly rounded, so monotone) is not below
// thr: sqrtf(x) < thr exactly where x < square_gate(thr).
float square_gate(float thr) {
  float x = thr * thr;
  while (x > 0.0f && sqrtf(x) >= thr) x = nextafterf(x, 0.0f);
  while (sqrtf(x) < thr) x = nextafterf(x, INFINITY);
  return x;
}

IcpArgs level_args(const kf_tracker* t, int l, const kf_frame_maps& live, const kf_frame_maps& model) {
  IcpArgs a = {};
  const kf_level_maps& L = live.level[l];
  const kf_level_maps& M = model.level[l];
  kf_intrinsics kl = kf_intrinsics_level(&t->k0, l);
  a.lvx = L.vx; a.lvy = L.vy; a.lvz = L.vz; a.lnx = L.nx; a.lny = L.ny; a.lnz = L.nz;
  a.mvx = M.vx; a.mvy = M.vy; a.mvz = M.vz; a.mnx = M.nx; a.mny = M.ny; a.mnz = M.nz;
  a.W = kl.width;
  a.H = kl.height;
  a.fx = kl.fx;
  a.fy = kl.fy;
  a.cx = kl.cx;
  a.cy = kl.cy;
  a.dist_thr2 = square_gate(t->params.dist_thresh_m);
  a.cos_thr = (float)cos((double)t->params.normal_thresh_deg * 3.14159265358979323846 / 180.0);
  a.partials = t->d_partials;
  a.ctrl = t->d_ctrl;
  a.level = l;
  return a;
}

static_assert(StepShape<0, 1>::kPixels == kShapePixels[0] && StepShape<1, 0>::kPixels == kShapePixels[1] &&
                  StepShape<2, 1>::kPixels == kShapePixels[2] && StepShape<3, 0>::kPixels == kShapePixels[3],
              "step shapes");

template <bool COMP>
void launch_step(int shape, int blocks, hipStream_t s, const IcpArgs& a, const StepArgs& S) {
  auto kern = shape == 0 ? icp_step<COMP, 0, 1> : shape == 1 ? icp_step<COMP, 1, 0> : shape == 2 ? icp_step<COMP, 2, 1>
                                                                                                : icp_step<COMP, 3, 0>;
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(kStepThreads), 0, s, a, S);
}

int level_blocks(const kf_tracker* t, int W, int H, int l) {
  const int ppt = (l == 0) ? 2 : 1;
  int b = div_up(W * H, kThreads * ppt);
  return b < t->max_blocks ? b : t->max_blocks;
}

kf_status check_maps(const kf_tracker* t, const kf_frame_maps& live, const kf_frame_maps& model,
                     int levels) {
  KF_CHECK_ARG(live.levels >= levels && model.levels >= levels, "maps have fewer levels than ICP");
  for (int l = 0; l < levels; ++l) {
    kf_intrinsics kl = kf_intrinsics_level(&t->k0, l);
    const kf_level_maps& L = live.level[l];
    const kf_level_maps& M = model.level[l];
    KF_CHECK_ARG(L.width == kl.width && L.height == kl.height, "live level size mismatch");
    KF_CHECK_ARG(M.width == kl.width && M.height == kl.height, "model level size mismatch");
    KF_CHECK_ARG(L.vx && L.vy && L.vz && L.nx && L.ny && L.nz, "live plane is NULL");
    KF_CHECK_ARG(M.vx && M.vy && M.vz && M.nx && M.ny && M.nz, "model plane is NULL");
  }
  return KF_OK;
}

}  // namespace

kf_status launch_icp_track(kf_tracker* t, const kf_frame_maps& live, const kf_frame_maps& model,
                           const kf_pose* d_guess, kf_pose* d_out, kf_icp_stats* d_stats,
                           hipStream_t s, bool single_launch, const IcpGate* gate, const FrameEnd* frame_end) {
  KF_CHECK_ARG(d_guess && d_out, "guess/out pose is NULL");
  const kf_icp_params& p = t->params;
  KF_TRY(check_maps(t, live, model, p.levels));
  kf_icp_stats* st = t->d_stats_tmp;
  double* slots[2] = {t->d_partials, t->d_partials + (size_t)t->max_blocks * kSlot};
  if (single_launch || p.single_launch) {
    ChainArgs C = {};
    C.levels = p.levels;
    int grid = 1;
    for (int l = 0; l < p.levels; ++l) {
      C.lv[l] = level_args(t, l, live, model);
      C.iters[l] = p.iterations[l];
      const int pixels = C.lv[l].W * C.lv[l].H;
      C.blocks[l] = step_blocks(pixels, t->max_blocks);
      C.shape[l] = step_shape(pixels);
      if (C.iters[l] > 0) grid = std::max(grid, chain_blocks(pixels, l, t->max_blocks));
    }
    if (t->chain_capacity < 0) {  // blocks of this kernel that can be resident at once
      int dev = 0, per_cu = 0, cus = 0;
      KF_HIP(hipGetDevice(&dev));
      KF_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
      if (p.compensated)
        KF_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, icp_chain<true>, kStepThreads, 0));
      else
        KF_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, icp_chain<false>, kStepThreads, 0));
      t->chain_capacity = per_cu * cus;
    }
    KF_CHECK_ARG(t->chain_capacity >= 1, "single-launch ICP cannot be resident on this device");
    if (grid > t->chain_capacity) grid = t->chain_capacity;
    C.guess = d_guess;
    C.out = d_out;
    C.slots[0] = slots[0];
    C.slots[1] = slots[1];
    C.user = d_stats;
    C.st = st;
    C.ctrl = t->d_ctrl;
    C.gate = gate ? *gate : IcpGate{};
    C.gated = gate ? 1 : 0;
    C.fe = frame_end ? *frame_end : FrameEnd{};
    C.fe_on = frame_end ? 1 : 0;
    if (p.compensated)
      hipLaunchKernelGGL(icp_chain<true>, dim3(grid), dim3(kStepThreads), 0, s, C);
    else
      hipLaunchKernelGGL(icp_chain<false>, dim3(grid), dim3(kStepThreads), 0, s, C);
    return check_launch("icp_chain");
  }
  StepArgs S = {};
  S.user = d_stats ? d_stats : st;  // the tracker's own statistics never carry the skip flag
  S.st = st;
  S.pose_in = d_guess;
  int step = 0, prev_blocks = 0, prev_level = 0;
  IcpArgs a = {};
  for (int l = p.levels - 1; l >= 0; --l) {
    a = level_args(t, l, live, model);
    const int blocks = step_blocks(a.W * a.H, t->max_blocks), shape = step_shape(a.W * a.H);
    for (int it = 0; it < p.iterations[l]; ++it, ++step) {
      S.first = step == 0 ? 1 : 0;
      S.index = step;
      S.pose_out = &t->d_work[step & 1];
      S.slots_in = slots[(step + 1) & 1];
      S.slots_out = slots[step & 1];
      S.nb_in = prev_blocks;
      S.level_in = prev_level;
      if (p.compensated) launch_step<true>(shape, blocks, s, a, S);
      else launch_step<false>(shape, blocks, s, a, S);
      KF_TRY(check_launch("icp_step"));
      S.pose_in = S.pose_out;
      prev_blocks = blocks;
      prev_level = l;
    }
  }
  S.slots_in = slots[(step + 1) & 1];
  S.nb_in = prev_blocks;
  S.level_in = prev_level;
  const IcpGate g = gate ? *gate : IcpGate{};
  const FrameEnd fe = frame_end ? *frame_end : FrameEnd{};
  hipLaunchKernelGGL(icp_finish, dim3(1), dim3(kSolveThreads), 0, s, a, S, step, d_out, d_stats, g,
                     gate ? 1 : 0, fe, frame_end ? 1 : 0);
  return check_launch("icp_finish");
}

kf_status launch_icp_reduce(kf_tracker* t, int level, const kf_frame_maps& live,
                            const kf_frame_maps& model, const kf_pose* d_est, double* d_sums,
                            uint8_t* d_mask, hipStream_t s) {
  KF_CHECK_ARG(level >= 0 && level < KF_MAX_LEVELS, "level out of range");
  KF_CHECK_ARG(d_est && d_sums, "pose/sums is NULL");
  KF_TRY(check_maps(t, live, model, level + 1));
  IcpArgs a = level_args(t, level, live, model);
  a.pose = const_cast<kf_pose*>(d_est);  // read only
  a.sums_out = d_sums;
  a.mask = d_mask;
  const int blocks = level_blocks(t, a.W, a.H, level);
  if (t->params.compensated)
    hipLaunchKernelGGL(icp_partials<true>, dim3(blocks), dim3(kThreads), 0, s, a);
  else
    hipLaunchKernelGGL(icp_partials<false>, dim3(blocks), dim3(kThreads), 0, s, a);
  KF_TRY(check_launch("icp_partials(reduce)"));
  hipLaunchKernelGGL(icp_sums, dim3(1), dim3(kSolveThreads), 0, s, a, blocks);
  return check_launch("icp_sums(reduce)");
}

kf_status launch_pose_constant_velocity(const kf_pose* d_prev2, const kf_pose* d_prev1,
                                        kf_pose* d_guess, hipStream_t s) {
  KF_CHECK_ARG(d_prev2 && d_prev1 && d_guess, "pose is NULL");
  hipLaunchKernelGGL(pose_const_velocity, dim3(1), dim3(64), 0, s, d_prev2, d_prev1, d_guess);
  return check_launch("pose_const_velocity");
}

kf_status launch_pose_copy(const kf_pose* d_src, kf_pose* d_dst, hipStream_t s) {
  hipLaunchKernelGGL(pose_copy, dim3(1), dim3(64), 0, s, d_src, d_dst);
  return check_launch("pose_copy");
}



// ---------------------------------------------------------------------------
// Tracking without allocation (kf_icp_track_noalloc).  The scratch a tracker
// allocates — two sets of block slots, the control block, the two alternating step
// poses and the statistics — lives in a file-scope device array, `scratch`.  Each
// device holds its own copy at its own address: the address is taken once per
// device with hipGetSymbolAddress (with that device current) and only that address
// is passed to kernels.  Every call on a device shares its copy, which keeps the
// last call's contents; the control block is cleared at the start of every call
// (by a kernel, so that the call can be captured into a graph).
namespace {

constexpr int kNoAllocSlots = KF_ICP_NOALLOC_MAX_SLOTS;
struct NoAllocScratch {
  double slots[2 * kNoAllocSlots * kSlot];
  kf_icp_ctrl ctrl;
  kf_pose work[2];
  kf_icp_stats stats;
};
static_assert(sizeof(NoAllocScratch) <= 300 * 1024, "no-allocation scratch larger than stated");

__device__ __align__(256) unsigned char scratch[sizeof(NoAllocScratch)];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
NoAllocScratch* g_scratch[kMaxDevices] = {};

// The current device's copy of `scratch` (its address taken on the first call).
kf_status scratch_of_current_device(NoAllocScratch** out) {
  int dev = 0;
  KF_HIP(hipGetDevice(&dev));
  KF_CHECK_ARG(dev >= 0 && dev < kMaxDevices, "device index beyond the no-allocation table");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch[dev]) {
    void* ptr = nullptr;
    KF_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    g_scratch[dev] = static_cast<NoAllocScratch*>(ptr);
  }
  *out = g_scratch[dev];
  return KF_OK;
}

__global__ void clear_ctrl(kf_icp_ctrl* c) {
  static_assert(sizeof(kf_icp_ctrl) % 4 == 0, "control block size");
  for (unsigned i = threadIdx.x; i < sizeof(kf_icp_ctrl) / 4; i += blockDim.x) reinterpret_cast<int*>(c)[i] = 0;
}

}  // namespace

kf_status launch_icp_track_noalloc(const kf_intrinsics& k0, const kf_icp_params& p, const kf_frame_maps& live,
                                   const kf_frame_maps& model, const kf_pose* d_guess, kf_pose* d_out,
                                   kf_icp_stats* d_stats, hipStream_t s) {
  // Images beyond 512 slots of three pixels a thread (one below the finest level) are
  // rejected: a step grid of more blocks than slots would have to be capped, which changes
  // the block partition and the sums' rounding.
  for (int l = 0; l < p.levels; ++l) {
    if (p.iterations[l] == 0) continue;
    const kf_intrinsics kl = kf_intrinsics_level(&k0, l);
    KF_CHECK_ARG(kl.width * kl.height <= kNoAllocSlots * kStepThreads * (l == 0 ? 3 : 1),
                 "image too large for kf_icp_track_noalloc (level-0 images up to 786432 pixels)");
  }
  NoAllocScratch* sc = nullptr;
  KF_TRY(scratch_of_current_device(&sc));
  kf_tracker t;  // a tracker handle over the scratch: nothing is allocated
  t.k0 = k0;
  t.params = p;
  t.max_blocks = kNoAllocSlots;
  t.d_partials = sc->slots;
  t.d_ctrl = &sc->ctrl;
  t.d_work = sc->work;
  t.d_stats_tmp = &sc->stats;
  t.chain_capacity = -1;
  hipLaunchKernelGGL(clear_ctrl, dim3(1), dim3(64), 0, s, &sc->ctrl);
  KF_TRY(check_launch("clear_ctrl"));
  return launch_icp_track(&t, live, model, d_guess, d_out, d_stats, s);
}

}  // namespace kf
