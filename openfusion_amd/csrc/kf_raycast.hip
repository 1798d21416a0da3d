// kf_raycast.hip — ray-marching raycaster over the TSDF volume.
//
// Replaces d_raycast / Raycaster::Raycast (Source/src/Raycaster.cu:97-242).  The
// reference marches 1.5 mm steps with nearest-voxel reads and takes the first
// voxel with tsdf <= 0 (Raycaster.cu:152-188); this kernel implements the
// trilinear sampling and linear zero-crossing refinement that the reference's
// disabled getSurfaceVertex intended (Raycaster.cu:287-350), with a two-speed
// march (step_far*T in free space, step_near voxels inside the truncation band)
// and trilinear central-difference gradient normals (the reference's
// getRenderedNormal, Raycaster.cu:64-94, takes central differences of voxels).
//
// The march runs in grid coordinates: g(t) = go + t * gd with go the camera
// centre and gd the ray direction in voxel units, one fused multiply-add per axis
// and sample; g = floor(g) + fract(g) gives the trilinear cell and weights.
//
// Ray/tile mapping: each wavefront of a 256-thread block takes an 8x8 pixel tile (rays
// in a wave stay coherent in the volume), the four together or a quarter of the image
// apart.  Block ids are remapped so that each of the 8 XCDs (which receive blocks
// round-robin) owns contiguous bands of tiles and its L2 sees neighbouring rays.
//
// Normals are computed once per wavefront after every ray of it has finished its
// march: each hit loads the 32 voxels of its six central-difference samples in one
// round of row loads.
//
// What bounds it: issue.  A round of the march is ~225 vector instructions (FP16
// records) at four cycles each, a wave makes ~9 rounds and its longest ray up to 20, and
// 4,800 waves of a 640x480 image share 1,024 SIMDs; then the latency of the longest
// waves' rounds, which end alone (vector pipes busy 57% of the kernel before the
// instruction counts below were cut, 39% of a wave's time in memory waits).  Hence: no
// domain check per sample, differences of FP16 halves without conversions, one face per
// axis in the free-space skip, no division inside the loop.  The time depends on the scene
// and the pose.  With the brick distances, over seven rooms: 512^3 FP16 at 640x480 37..68 us
// before, 31..56 now (the first room 43.0 and 34.8); 256^3 FP32 at 319x241 23..42 and 20..36.
// (One of 35 rooms and sizes is slower, by the spread below: 768^3 FP16 at 640x480 49 -> 54.)
// Looking at the map once per sample and loading corners only where a brick
// is set (fewer instructions a round, more rounds), corner loads ahead of the map's
// answer, four or five samples a round, and a wave priority that grows with its rounds
// were all slower.
#include <hip/hip_ext.h>

#include <type_traits>

#include "kf_device.hpp"
#include "kf_internal.hpp"

namespace kf {
namespace {

constexpr int kXcds = 8;
// Long rays lie together in the image, and the waves of a block share a CU's L1, whose
// line lookups a round of corner loads takes 800 of: from 384 blocks (1.5 a CU) on, a
// block's four tiles are a quarter of the image apart.  512^3 FP16 over seven rooms,
// together / apart: 480x360 28.8..48.8 / 25.5..48.5 us, 640x480 31.5..64.4 / 31.5..56.4,
// 800x600 41.4..80.2 / 43.2..67.3, each room between 16 % faster and 5 % slower apart; late
// in a 300-frame stream, beside the frame's other kernels, 4,496 / 4,568 frames/s.  With
// about a block a CU there is nothing to balance and the tiles' shared lines count: 256^3
// FP32 at 319x241 19.6..36.1 / 19.8..33.7, the cheap rooms slower, the dear ones faster.
constexpr int kSpreadBlocks = 384;

struct RayArgs {
  const void* vox;
  const kf_pose* pose;
  kf_level_maps out;
  // model pyramid: level l >= 1 takes every 2^l-th sample of level 0, written by the
  // lane of that level-0 pixel
  kf_level_maps sub[KF_MAX_LEVELS];  // [1], [2] used
  int levels;
  unsigned long long* steps;
  unsigned long long* diag;  // optional [samples that loaded corners, batches, skipped steps, 64 x wave max
                             // batches, max batches of a ray]
  const uint8_t* bdist;           // brick distances to the nearest set brick, 0 = set (NULL: no map)
  int occ_nb;                     // bricks per axis
  int occ_words;                  // 64-bit occupancy words per brick column
  int n;
  float h, inv_h, ox, oy, oz;
  float fx, fy, cx, cy;
  int W, H;
  float min_depth, step_far_m, step_near_m;
  float inv_step_far;  // 1 / step_far_m (estimates only)
  int max_steps;
  int blocks_x, blocks_y;
  int spread;  // a block's wavefronts take tiles a quarter of the image apart
};

// Interpolations and points along a ray are fused multiply-adds (one rounding each;
// the oracle computes them the same way).
__device__ __forceinline__ float lerp(float a, float b, float t) { return fmaf(b - a, t, a); }
__device__ __forceinline__ f3 ray_at(f3 o, f3 d, float t) { return f3{fmaf(t, d.x, o.x), fmaf(t, d.y, o.y), fmaf(t, d.z, o.z)}; }

// Byte offset of voxel (ix, iy, iz) in the x-major volume.  OFF32: the volume's
// byte size fits in 32 bits, so the offset is one 32-bit register (24-bit
// multiplies, exact for n <= 1024) and every load below is a uniform base address
// plus that register.
template <bool OFF32>
using voff_t = typename std::conditional<OFF32, unsigned, size_t>::type;

template <int FMT, bool OFF32>
__device__ __forceinline__ voff_t<OFF32> vox_offset(int n, int ix, int iy, int iz) {
  constexpr unsigned kB = FMT == KF_VOXEL_F16 ? 4u : 8u;
  if constexpr (OFF32) {
    const unsigned un = (unsigned)n;
    const unsigned row = opaque_u32(__umul24((unsigned)ix, un) + (unsigned)iy);
    return opaque_u32(__umul24(row, un) + (unsigned)iz) * kB;
  } else {
    return ((((size_t)ix * (size_t)n) + (size_t)iy) * (size_t)n + (size_t)iz) * kB;
  }
}

// The eight corners of the trilinear cell whose base voxel is at byte offset o.
// The (z, z+1) pairs are adjacent records, fetched by one load each: 8 bytes for
// FP16 records, 16 bytes ({f, w} twice) for FP32 records.
typedef unsigned int u32x2_a4 __attribute__((ext_vector_type(2), aligned(4)));
typedef unsigned int u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x4_a8 __attribute__((ext_vector_type(4), aligned(8)));

template <int FMT>
using pair_ld = typename std::conditional<FMT == KF_VOXEL_F16, u32x2_a4, f32x4_a8>::type;
template <int FMT>
struct Corners {  // the (z, z + 1) pairs at (x, y), (x, y + 1), (x + 1, y), (x + 1, y + 1)
  pair_ld<FMT> q[4];
};

template <int FMT, bool OFF32>
__device__ __forceinline__ Corners<FMT> load_corners(const RayArgs& a, voff_t<OFF32> o) {
  constexpr unsigned kB = FMT == KF_VOXEL_F16 ? 4u : 8u;
  // an opaque 32-bit register keeps the base-register + 32-bit-offset load form
  if constexpr (OFF32) o = opaque_u32(o);
  const char* b[4];
  b[0] = static_cast<const char*>(a.vox);
  b[1] = b[0] + (size_t)a.n * kB;        // y + 1
  b[2] = b[0] + (size_t)a.n * a.n * kB;  // x + 1
  b[3] = b[2] + (size_t)a.n * kB;        // x + 1, y + 1
  Corners<FMT> c;
#pragma unroll
  for (int i = 0; i < 4; ++i) c.q[i] = *reinterpret_cast<const pair_ld<FMT>*>(b[i] + o);
  return c;
}

// lerp of the FP16 halves of two voxel records, converted as they are read: b - a and
// fma(b - a, t, a), each one rounding to FP32, as lerp() of the converted values (the
// difference is written as fma(b, 1, -a); two instructions instead of four).
__device__ __forceinline__ float lerp_h(uint32_t a, uint32_t b, float t) {
  float d, r;
  asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel_hi:[1,0,1]" : "=v"(d) : "v"(b), "v"(a));
  asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[0,0,1]" : "=v"(r) : "v"(d), "v"(t), "v"(a));
  return r;
}

// Trilinear value from four values interpolated along z and the x and y fractions.
__device__ __forceinline__ float bilinear(float c00, float c01, float c10, float c11, float tx, float ty) {
  return lerp(lerp(c00, c01, ty), lerp(c10, c11, ty), tx);
}
template <int FMT>
__device__ __forceinline__ float trilinear(const Corners<FMT>& c, float tx, float ty, float tz) {
  float z[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (FMT == KF_VOXEL_F16)
      z[i] = lerp_h(c.q[i].x, c.q[i].y, tz);
    else
      z[i] = lerp(c.q[i].x, c.q[i].z, tz);
  }
  return bilinear(z[0], z[1], z[2], z[3], tx, ty);
}

// Inside the trilinear domain: every coordinate in [0, n - 1).
__device__ __forceinline__ bool in_domain(f3 g, float lim) {
  return fminf(fminf(g.x, g.y), g.z) >= 0.0f && fmaxf(fmaxf(g.x, g.y), g.z) < lim;
}

// Whether any lane's condition holds (the lane mask itself, no vector compare).
__device__ __forceinline__ bool any_lane(bool c) { return __builtin_amdgcn_ballot_w64(c) != 0; }

// K trilinear samples of f at grid points g[j]: 1 where ok[j] is false (a point outside
// the trilinear domain, or one that the march does not reach).  Base voxel floor(g),
// weights g - floor(g).  When the brick of the base voxel is clear in the occupancy map
// (its brick distance is not 0), all eight corners hold f == 1 and the interpolation is
// exactly 1 (a + (b - a) t with a = b = 1), so the voxel loads are skipped: the value is
// the same.  dclear (optional): the brick distance of each sample whose brick is clear
// (>= 1), 0 otherwise.  Three phases, so that a batch costs about one map latency plus
// one voxel latency instead of K of each: the distance bytes of all samples, then the
// corners of all samples (one wave-uniform branch; lanes whose sample needs no corners
// read voxel 0 instead, which stays cached), then the interpolations.  use_map = false:
// this lane loads the corners without looking at the map (dclear 0).  need: the samples
// that loaded corners.
template <int FMT, bool OFF32, int K>
__device__ __forceinline__ void sample_points(const RayArgs& a, const f3* g, const bool* ok, float* fk, bool* need,
                                              int* dclear = nullptr, bool use_map = true) {
  // positions are finite (finite pose, t inside the slab interval); offsets of samples
  // with ok false are not used
  int d[K];
#pragma unroll
  for (int j = 0; j < K; ++j) d[j] = 0;
  const bool map_lane = a.bdist != nullptr && use_map;
  if (any_lane(map_lane)) {  // uniform
    // the brick's distance byte (64 per occupancy word of the column): 0 for a set
    // brick (its bit in the occupancy map), else the distance to the nearest set one;
    // lanes that do not use the map load the corners whatever the brick
    const unsigned row = (unsigned)kOccWordBricks * (unsigned)a.occ_words;
    unsigned o[K];
#pragma unroll
    for (int j = 0; j < K; ++j) {
      const int bx = (int)g[j].x >> 3, by = (int)g[j].y >> 3, bz = (int)g[j].z >> 3;
      const unsigned col = opaque_u32(__umul24((unsigned)bx, (unsigned)a.occ_nb) + (unsigned)by);
      o[j] = opaque_u32(__umul24(col, row) + (unsigned)bz);
      o[j] = ok[j] && map_lane ? o[j] : 0u;
    }
#pragma unroll
    for (int j = 0; j < K; ++j) d[j] = a.bdist[opaque_u32(o[j])];
#pragma unroll
    for (int j = 0; j < K; ++j) d[j] = ok[j] && map_lane ? d[j] : 0;
  }
  bool any = false;
#pragma unroll
  for (int j = 0; j < K; ++j) {
    need[j] = ok[j] && d[j] == 0;
    fk[j] = 1.0f;
    any = any || need[j];
    if (dclear) dclear[j] = d[j];
  }
  if (any_lane(any)) {
    Corners<FMT> c[K];
#pragma unroll
    for (int j = 0; j < K; ++j) {
      const voff_t<OFF32> o = vox_offset<FMT, OFF32>(a.n, (int)g[j].x, (int)g[j].y, (int)g[j].z);
      c[j] = load_corners<FMT, OFF32>(a, need[j] ? o : (voff_t<OFF32>)0);
    }
#pragma unroll
    for (int j = 0; j < K; ++j) {
      // g >= 0 where needed, so fract(g) = g - floor(g) = g - (float)(int)g exactly
      const float v = trilinear(c[j], __builtin_amdgcn_fractf(g[j].x), __builtin_amdgcn_fractf(g[j].y),
                                __builtin_amdgcn_fractf(g[j].z));
      fk[j] = need[j] ? v : 1.0f;
    }
  }
}

// Grid position of ray parameter t.
__device__ __forceinline__ f3 gpos(f3 go, f3 gd, float t) {
  return f3{fmaf(t, gd.x, go.x), fmaf(t, gd.y, go.y), fmaf(t, gd.z, go.z)};
}

// The six central-difference samples at grid point gh (x+1, x-1, y+1, y-1, z+1, z-1)
// for every lane with `want`.  Returns whether all six are inside the trilinear domain
// (false without `want`).  Their 48 corners are 32 voxels in 12 z-rows around the base
// voxel b of gh: (z-1 .. z+2) of the four rows (x, y), (x, y+1), (x+1, y), (x+1, y+1),
// and (z, z+1) of the rows next to them along x and y.  The lane loads each row once
// (FP16 records: one 16-byte or one 8-byte load, 12 in flight together): no pass
// through LDS, no wave reduction and no index division.  (The wave's samples staged as a
// box in LDS took ~550 vector instructions and a chain of reductions where this takes
// ~150: 39.6 -> 37.3 us with the brick distances at 512^3 FP16, 32.1 -> 30.5 at 256^3.)
template <int FMT, bool OFF32>
__device__ __forceinline__ bool gradient_samples(const RayArgs& a, bool want, f3 gh, float* fq) {
  constexpr unsigned kB = FMT == KF_VOXEL_F16 ? 4u : 8u;
  const float lim = (float)(a.n - 1);
  const f3 q[6] = {f3{gh.x + 1.0f, gh.y, gh.z}, f3{gh.x - 1.0f, gh.y, gh.z}, f3{gh.x, gh.y + 1.0f, gh.z},
                   f3{gh.x, gh.y - 1.0f, gh.z}, f3{gh.x, gh.y, gh.z + 1.0f}, f3{gh.x, gh.y, gh.z - 1.0f}};
  // rounding is monotone, so these six coordinates bound the others
  const bool all = want && fminf(fminf(q[1].x, q[3].y), q[5].z) >= 0.0f && fmaxf(fmaxf(q[0].x, q[2].y), q[4].z) < lim;
  const int bx = all ? (int)gh.x : 0, by = all ? (int)gh.y : 0, bz = all ? (int)gh.z : 0;
  // gh + 1 can round up to the next whole number where the exponent changes: its base
  // voxel is then not b + 1.  Such a wave takes the samples one by one.
  const bool plain = !all || ((int)q[0].x == bx + 1 && (int)q[1].x == bx - 1 && (int)q[2].y == by + 1 &&
                              (int)q[3].y == by - 1 && (int)q[4].z == bz + 1 && (int)q[5].z == bz - 1);
  if (any_lane(!plain)) {
    const bool okq[3] = {all, all, all};
    bool need[3];
    sample_points<FMT, OFF32, 3>(a, q, okq, fq, need);
    sample_points<FMT, OFF32, 3>(a, q + 3, okq, fq + 3, need);
  } else if (all) {
    typedef pair_ld<FMT> pair_t;
    voff_t<OFF32> o = vox_offset<FMT, OFF32>(a.n, bx, by, bz);
    if constexpr (OFF32) o = opaque_u32(o);
    const ptrdiff_t sy = (ptrdiff_t)a.n * kB, sx = sy * a.n;
    auto row = [&](ptrdiff_t off) { return static_cast<const char*>(a.vox) + off + o; };
    struct Row {
      pair_t m, p;  // (z - 1, z), (z + 1, z + 2)
    } r[4];         // (x, y), (x, y + 1), (x + 1, y), (x + 1, y + 1)
    pair_t xm[2], xp[2], ym[2], yp[2];  // (z, z + 1) at x - 1 and x + 2 (y, y + 1), at y - 1 and y + 2 (x, x + 1)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const char* p = row((i >> 1) * sx + (i & 1) * sy - (ptrdiff_t)kB);
      if constexpr (FMT == KF_VOXEL_F16) {
        const u32x4_a4 w = *reinterpret_cast<const u32x4_a4*>(p);
        r[i].m = pair_t{w.x, w.y};
        r[i].p = pair_t{w.z, w.w};
      } else {
        r[i].m = *reinterpret_cast<const f32x4_a8*>(p);
        r[i].p = *reinterpret_cast<const f32x4_a8*>(p + 2 * kB);
      }
    }
    auto pair = [&](ptrdiff_t off) { return *reinterpret_cast<const pair_ld<FMT>*>(row(off)); };
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      xm[i] = pair(i * sy - sx);
      xp[i] = pair(i * sy + 2 * sx);
      ym[i] = pair(i * sx - sy);
      yp[i] = pair(i * sx + 2 * sy);
    }
    // (z, z + 1) of a central row
    auto mid = [&](int i) {
      if constexpr (FMT == KF_VOXEL_F16)
        return pair_t{r[i].m.y, r[i].p.x};
      else
        return pair_t{r[i].m.z, r[i].m.w, r[i].p.x, r[i].p.y};
    };
    auto take = [&](int j, pair_t c00, pair_t c01, pair_t c10, pair_t c11) {
      const Corners<FMT> c{{c00, c01, c10, c11}};
      fq[j] = trilinear(c, __builtin_amdgcn_fractf(q[j].x), __builtin_amdgcn_fractf(q[j].y),
                        __builtin_amdgcn_fractf(q[j].z));
    };
    take(0, mid(2), mid(3), xp[0], xp[1]);
    take(1, xm[0], xm[1], mid(0), mid(1));
    take(2, mid(1), yp[0], mid(3), yp[1]);
    take(3, ym[0], mid(0), ym[1], mid(2));
    take(4, r[0].p, r[1].p, r[2].p, r[3].p);
    take(5, r[0].m, r[1].m, r[2].m, r[3].m);
  }
  return all;
}

template <int FMT, bool OFF32>
__global__ __launch_bounds__(256) void raycast(RayArgs a) {
  // XCD-aware block remap: logical = (xcd band) + (position within band).
  const int nb = a.blocks_x * a.blocks_y;
  const int per = (nb + kXcds - 1) / kXcds;
  const int xcd = blockIdx.x % kXcds, slot = blockIdx.x / kXcds;
  const int logical = xcd * per + slot;
  if (logical >= nb) return;  // whole block
  const int by = logical / a.blocks_x, bx = logical - by * a.blocks_x;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  int x = bx * 16 + (wave & 1) * 8, y = by * 16 + (wave >> 1) * 8;
  if (a.spread) {
    const int tile = logical + wave * nb, tx = 2 * a.blocks_x;
    x = tile % tx * 8;
    y = tile / tx * 8;
  }
  x += lane & 7;
  y += lane >> 3;
  const bool active = x < a.W && y < a.H;  // no early return: the step count is wave-reduced
  const int idx = active ? y * a.W + x : 0;
  const kf_posef P = a.pose->wc;

  const float xn = ((float)x - a.cx) / a.fx;
  const float yn = ((float)y - a.cy) / a.fy;
  const f3 dw = rot(P.r, f3{xn, yn, 1.0f});
  const float len = sqrtf(dot(dw, dw));
  const float il = 1.0f / len;
  const f3 dir = f3{dw.x * il, dw.y * il, dw.z * il};
  const f3 o = f3{P.t[0], P.t[1], P.t[2]};
  // the ray in grid coordinates: g(t) = go + t gd
  const f3 go = f3{fmaf(o.x - a.ox, a.inv_h, -0.5f), fmaf(o.y - a.oy, a.inv_h, -0.5f),
                   fmaf(o.z - a.oz, a.inv_h, -0.5f)};
  const f3 gd = f3{dir.x * a.inv_h, dir.y * a.inv_h, dir.z * a.inv_h};

  // Slab test against the voxel-centre box shrunk by 0.01 voxel, so that the first
  // and last samples fall strictly inside the trilinear domain despite rounding.
  const float lo = 0.51f * a.h, hi = ((float)a.n - 0.51f) * a.h;
  const float blo[3] = {a.ox + lo, a.oy + lo, a.oz + lo};
  const float bhi[3] = {a.ox + hi, a.oy + hi, a.oz + hi};
  const float oo[3] = {o.x, o.y, o.z}, dd[3] = {dir.x, dir.y, dir.z};
  float tnear = a.min_depth * len, tfar = 3.0e38f;
  bool hit = true;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    if (dd[k] != 0.0f) {
      const float t1 = (blo[k] - oo[k]) / dd[k];
      const float t2 = (bhi[k] - oo[k]) / dd[k];
      tnear = fmaxf(tnear, fminf(t1, t2));
      tfar = fminf(tfar, fmaxf(t1, t2));
    } else if (!(oo[k] >= blo[k] && oo[k] <= bhi[k])) {
      hit = false;
    }
  }
  int nsteps = 0;
  int n_loads = 0, n_batches = 0, n_skipped = 0;  // diagnostics (stage-timing mode)
  bool found = false;  // a zero crossing, refined to ray parameter ts
  float ts = 0.0f;
  if (active && hit && tnear < tfar) {
    // The march: step_far while the last sample is +1 (free space), step_near
    // otherwise; stop at the first sample < 0, outside the domain, past tfar or
    // after max_steps.  Positions are counted per segment of equal steps: from the
    // segment's start t0 the i-th step is at fma(i, step, t0), and a segment starts
    // where the step size changes.  Samples are fetched kSpec at a time assuming the
    // step size stays the same and then consumed in order; a batch ends where the
    // march would change step size or stop, so the result and the step count equal
    // the one-step-at-a-time march while the dependent-load chain is up to kSpec
    // times shorter.  FP16 records: three samples a batch (80 VGPRs, six waves per
    // SIMD) as fast as two (70 VGPRs: 35.6 and 34.8 us) when the image is alone on the
    // chip, and ahead once the frame's concurrent kernels share it.  FP32 records
    // (16-byte corner loads): three would need 110 VGPRs (four waves per SIMD, fewer
    // than the 4,800 waves), so two.
    constexpr int kSpec = FMT == KF_VOXEL_F16 ? 3 : 2;
    const float lim = (float)(a.n - 1);
    float t = tnear, fp;
    bool ok;
    int last_d;  // brick distance of the sample at t when its brick is clear, else 0
    {
      const f3 g0 = gpos(go, gd, t);
      ok = in_domain(g0, lim);
      bool need;
      sample_points<FMT, OFF32, 1>(a, &g0, &ok, &fp, &need, &last_d);
      // A coordinate of g(t) is a monotone function of t, so the part of [tnear, tfar]
      // whose points are in the domain is an interval from tnear on: with its end as
      // tfar (tfar itself but for rounding far outside the volume; else bisected), the
      // march needs no domain check.
      if (ok && !in_domain(gpos(go, gd, tfar), lim)) {
        float in = tnear;
        for (int k = 0; k < 256; ++k) {
          const float mid = in + (tfar - in) * 0.5f;
          if (!(mid > in && mid < tfar)) break;
          const bool inside = in_domain(gpos(go, gd, mid), lim);
          in = inside ? mid : in;
          tfar = inside ? tfar : mid;
        }
        tfar = in;
      }
      ok = ok && fp >= 0.0f;
    }
    float t0 = t;           // start of the current segment
    int i = 0;              // steps taken in it
    int imax = a.max_steps;  // steps that may still be taken at its start
    float fb = 0.0f;         // the sample that ended the march in a crossing
    bool seg_far = fp >= 1.0f;
    // Free-space skip.  From a far-mode position t (sample 1) whose base voxel lies
    // in a brick at distance D >= 1 from the nearest set brick, every brick within
    // D - 1 of it (a cube of 2D - 1 bricks) is clear, so every sample whose base
    // voxel lies in that box is exactly 1.  Advance k far steps at once: the k
    // positions are those of the segment, fma(i + 1 .. i + k, step, t0), and the grid
    // coordinate of a position is a monotone function of i on each axis, so if the
    // last one is still in the box (checked with the exact sample arithmetic) every
    // intermediate one is too.  The step count, the position and the value are those
    // of the step-by-step march.  A ray can leave the box only through the faces
    // ahead of it: axes along which it runs down are mirrored (sign and order of
    // floats negate exactly; brick b becomes ~b), so each axis has one face, above.
    float gom[3], gdm[3], rd[3], rc[3], top[3];
    int flip[3];
    const float go_[3] = {go.x, go.y, go.z}, gd_[3] = {gd.x, gd.y, gd.z};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const bool down = gd_[k] < 0.0f;
      flip[k] = down ? -1 : 0;
      top[k] = down ? 0.0f : (float)(a.n - 1);
      gom[k] = down ? -go_[k] : go_[k];
      gdm[k] = fabsf(gd_[k]);
      // exit estimate of a face: face * rd + rc (not a number for an axis the ray does
      // not move along; the minimum below passes over it)
      rd[k] = __builtin_amdgcn_rcpf(gdm[k]);
      rc[k] = -gom[k] * rd[k];
    }
    auto skip_free = [&](int D) {
      const f3 gp = gpos(go, gd, t);
      const int b[3] = {(int)gp.x >> 3, (int)gp.y >> 3, (int)gp.z >> 3};
      float face[3], e[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        face[k] = fminf((float)(((b[k] ^ flip[k]) + D) * 8), top[k]);
        e[k] = fmaf(face[k], rd[k], rc[k]);
      }
      // Approximate exit parameter of the box: only the estimate of k depends on it, and
      // the skip is verified with the exact arithmetic below.
      const float te = fminf(fminf(tfar, e[0]), fminf(e[1], e[2]));
      int k = (int)fminf((te - t) * a.inv_step_far, (float)a.max_steps) - 1;
      k = min(k, imax - i);
      if (k <= 0) return;
      const float tt = fmaf((float)(i + k), a.step_far_m, t0);
      bool in = tt <= tfar;
#pragma unroll
      for (int k = 0; k < 3; ++k) in = in && fmaf(tt, gdm[k], gom[k]) < face[k];
      if (in) {
        t = tt;
        i += k;
        n_skipped += k;
      }
    };
    bool run = ok && i < imax;
    while (run) {
      const bool far = fp >= 1.0f;
      if (far != seg_far) {  // the step size changes: a new segment from t
        t0 = t;
        imax -= i;
        i = 0;
        seg_far = far;
      }
      if (far && last_d > 0) skip_free(last_d);
      const float st = far ? a.step_far_m : a.step_near_m;
      float tk[kSpec], fk[kSpec];
      f3 gk[kSpec];
      bool vk[kSpec];
      int ck[kSpec];
#pragma unroll
      for (int j = 0; j < kSpec; ++j) {
        tk[j] = fmaf((float)(i + j + 1), st, t0);
        gk[j] = gpos(go, gd, tk[j]);
        vk[j] = tk[j] <= tfar;
      }
      // Inside the truncation band (near mode) the bricks ahead hold the surface, so
      // the corners are loaded without the map's dependent lookup first: one memory
      // latency per batch instead of two (the values are the same; the map only
      // spares loads).
      bool lk[kSpec];
      sample_points<FMT, OFF32, kSpec>(a, gk, vk, fk, lk, ck, far);
      if (a.diag) {  // uniform
        ++n_batches;
#pragma unroll
        for (int j = 0; j < kSpec; ++j) n_loads += lk[j] ? 1 : 0;
      }
      // Consume the batch in order, as selects rather than branches.  Sample j is
      // examined when every earlier sample of the batch was consumed (valid, no
      // crossing) and kept the step size; then it is step i + j of the segment, taken
      // while i + j < imax.  A step that finds its sample invalid still counts and
      // ends the march; a crossing ends it with t and fp at the last consumed sample
      // (>= 0) and fb at this one (< 0).
      bool go_on = true;
      const int left = imax - i;
#pragma unroll
      for (int j = 0; j < kSpec; ++j) {
        const bool v = go_on && j < left && vk[j];
        const bool x = v && fk[j] < 0.0f;
        const bool c = v && !x;
        if (x) fb = fk[j];
        if (go_on && !c) run = false;
        go_on = c && ((fk[j] >= 1.0f) == far);
        if (c) {
          t = tk[j];
          fp = fk[j];
          last_d = ck[j];
          ++i;
        }
      }
      run = run && i < imax;
    }
    if (ok) nsteps = a.max_steps - (imax - i) + (i < imax ? 1 : 0);
    if (fb < 0.0f) {
      ts = t + (seg_far ? a.step_far_m : a.step_near_m) * (fp / (fp - fb));
      found = true;
    }
  }
  // Normals of the wave's hits: trilinear central differences at the refined point.
  f3 vert = f3{nanf_(), nanf_(), nanf_()}, nrm = vert;
  {
    const f3 gh = found ? gpos(go, gd, ts) : f3{0.0f, 0.0f, 0.0f};
    float fq[6];
    if (gradient_samples<FMT, OFF32>(a, found, gh, fq)) {
      const f3 gr = f3{fq[0] - fq[1], fq[2] - fq[3], fq[4] - fq[5]};
      const float gl = sqrtf(dot(gr, gr));
      if (gl > 0.0f) {
        const float ig = 1.0f / gl;
        nrm = f3{gr.x * ig, gr.y * ig, gr.z * ig};
        vert = ray_at(o, dir, ts);
      }
    }
  }
  if (active) {
    a.out.vx[idx] = vert.x;
    a.out.vy[idx] = vert.y;
    a.out.vz[idx] = vert.z;
    a.out.nx[idx] = nrm.x;
    a.out.ny[idx] = nrm.y;
    a.out.nz[idx] = nrm.z;
#pragma unroll
    for (int l = 1; l < KF_MAX_LEVELS; ++l) {
      const int m = (1 << l) - 1;
      if (l < a.levels && !(x & m) && !(y & m)) {
        const kf_level_maps& ol = a.sub[l];
        const int xl = x >> l, yl = y >> l;
        if (xl < ol.width && yl < ol.height) {
          const int j = yl * ol.width + xl;
          ol.vx[j] = vert.x;
          ol.vy[j] = vert.y;
          ol.vz[j] = vert.z;
          ol.nx[j] = nrm.x;
          ol.ny[j] = nrm.y;
          ol.nz[j] = nrm.z;
        }
      }
    }
  }
  if (a.diag) {  // diagnostics: one device atomic per block and counter
    __shared__ int dred[4][4];
    const int v0 = wave_sum_i_lane63(n_loads), v1 = wave_sum_i_lane63(n_batches), v2 = wave_sum_i_lane63(n_skipped);
    int mx = n_batches;  // the wave runs as long as its longest ray
    for (int off = 32; off > 0; off >>= 1) mx = max(mx, __shfl_xor(mx, off, kWave));
    if (lane == 63) {
      dred[0][wave] = v0;
      dred[1][wave] = v1;
      dred[2][wave] = v2;
      dred[3][wave] = mx * kWave;
    }
    __syncthreads();
    if (threadIdx.x < 4) {
      const int q = threadIdx.x;
      const int b = (dred[q][0] + dred[q][1]) + (dred[q][2] + dred[q][3]);
      if (b) atomicAdd(&a.diag[q], (unsigned long long)b);
    } else if (threadIdx.x == 4) {
      const int m = max(max(dred[3][0], dred[3][1]), max(dred[3][2], dred[3][3])) / kWave;
      atomicMax(&a.diag[4], (unsigned long long)m);
    }
  }
  if (a.steps) {  // one device atomic per block (uniform branch)
    __shared__ int red[4];
    const int tot = wave_sum_i_lane63(nsteps);
    if (lane == 63) red[wave] = tot;
    __syncthreads();
    if (threadIdx.x == 0) {
      const int b = (red[0] + red[1]) + (red[2] + red[3]);
      if (b) atomicAdd(a.steps, (unsigned long long)b);
    }
  }
}

}  // namespace

kf_status launch_raycast(const kf_volume* v, const kf_intrinsics& k0, const kf_raycast_params& p,
                         const kf_pose* d_pose, kf_frame_maps& model, unsigned long long* d_steps,
                         hipStream_t s, hipEvent_t after_distances, unsigned long long* d_diag,
                         hipEvent_t kernel_start, hipEvent_t kernel_stop) {
  KF_CHECK_ARG(d_pose != nullptr, "pose is NULL");
  KF_CHECK_ARG(model.levels >= 1 && model.levels <= KF_MAX_LEVELS, "model levels must be 1..3");
  KF_CHECK_ARG(p.step_far > 0.0f && p.step_near > 0.0f && p.max_steps > 0, "bad march steps");
  for (int l = 0; l < model.levels; ++l) {
    kf_intrinsics kl = kf_intrinsics_level(&k0, l);
    const kf_level_maps& m = model.level[l];
    KF_CHECK_ARG(m.width == kl.width && m.height == kl.height, "model level size mismatch");
    KF_CHECK_ARG(m.vx && m.vy && m.vz && m.nx && m.ny && m.nz, "model plane is NULL");
  }
  const kf_volume_desc& d = v->desc;
  RayArgs a;
  a.vox = v->d_voxels;
  a.pose = d_pose;
  a.out = model.level[0];
  a.levels = model.levels;
  for (int l = 0; l < KF_MAX_LEVELS; ++l) a.sub[l] = l < model.levels ? model.level[l] : kf_level_maps{};
  a.steps = d_steps;
  a.diag = d_diag;
  KF_TRY(ensure_occupancy(v, s));
  KF_TRY(launch_brick_distance(v, s));
  if (after_distances) KF_HIP(hipEventRecord(after_distances, s));
  a.bdist = v->occ_enabled ? v->d_bdist : nullptr;
  a.occ_nb = v->occ_nb;
  a.occ_words = v->occ_words;
  a.n = d.n;
  a.h = d.extent_m / (float)d.n;
  a.inv_h = (float)d.n / d.extent_m;
  a.ox = d.origin_m[0];
  a.oy = d.origin_m[1];
  a.oz = d.origin_m[2];
  a.fx = k0.fx;
  a.fy = k0.fy;
  a.cx = k0.cx;
  a.cy = k0.cy;
  a.W = k0.width;
  a.H = k0.height;
  a.min_depth = p.min_depth_m;
  a.step_far_m = p.step_far * d.trunc_m;
  a.step_near_m = p.step_near * a.h;
  a.inv_step_far = 1.0f / a.step_far_m;
  a.max_steps = p.max_steps;
  a.blocks_x = div_up(k0.width, 16);
  a.blocks_y = div_up(k0.height, 16);
  const int nb = a.blocks_x * a.blocks_y;
  const int grid = ((nb + kXcds - 1) / kXcds) * kXcds;
  a.spread = nb >= kSpreadBlocks;
  // 32-bit voxel offsets when every byte offset of the volume fits in 32 bits
  const bool off32 = v->bytes <= 0xffffffffull && d.n <= 1024;
  auto kern = d.format == KF_VOXEL_F16 ? (off32 ? raycast<KF_VOXEL_F16, true> : raycast<KF_VOXEL_F16, false>)
                                       : (off32 ? raycast<KF_VOXEL_F32, true> : raycast<KF_VOXEL_F32, false>);
  if (kernel_start && kernel_stop)
    hipExtLaunchKernelGGL(kern, dim3(grid), dim3(256), 0, s, kernel_start, kernel_stop, 0, a);
  else
    hipLaunchKernelGGL(kern, dim3(grid), dim3(256), 0, s, a);
  return check_launch("raycast");
}

}  // namespace kf
