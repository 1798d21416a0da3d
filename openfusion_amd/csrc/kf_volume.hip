// kf_volume.hip — TSDF volume initialisation and the projective integration sweep.
//
// Replaces d_initVoxelArray (Source/src/General.cu:27-50) and d_integrateVolume /
// VolumeIntegrator::Integrate (Source/src/VolumeIntegrator.cu:86-201).
//
// Layout: voxel (x,y,z) at index (x*n + y)*n + z (z fastest), one 8-byte {f, w}
// (FP32) or one 4-byte {half f, u16 w} (FP16) word per voxel, f = tsdf/T.
//
// The sweep reads and writes only voxels that are updated, and runs the exact
// per-voxel test only where its outcome is not known for a whole brick:
//   1. raylen_tiles: min / max raylen of every 8x8 and 32x32 pixel tile.
//   2. brick_classify: one thread per 8^3 brick projects the brick's corner voxel
//      centres in FP64 and, from the tile extrema under its footprint, marks it
//      skip (no voxel can be updated), free (every voxel is updated with f = 1) or
//      exact, with margins far above the FP32 error of the per-voxel test.
//      Exact bricks are appended to the front of a work list, free ones to its back.
//   3. integrate: a wavefront takes one listed brick at a time (waves stride over
//      the exact bricks, then the free ones, so each gets an even share of the
//      costlier exact bricks), a lane per (y, z) of the brick and the eight x-slices
//      together:
//      free bricks update every voxel with f = 1, exact bricks evaluate the FP32
//      test of the reference's per-voxel body (in metres, z-forward camera) per
//      voxel.  A voxel is stored only if its bits change.  Skip, free and exact give
//      each voxel the outcome of the per-voxel test, so voxels, update masks and
//      counts are those of testing every voxel.
#include <hip/hip_ext.h>

#include <type_traits>

#include "kf_device.hpp"
#include "kf_internal.hpp"
#include "kf_launch.hpp"

namespace kf {
namespace {

constexpr int kWavesPerBlock = 4;
constexpr int kSweepMaxBlocks = 4096;  // 16384 waves: two full waves of residency on 256 CUs
// The sweep's blocks (their waves stride over the brick list): more than can be
// resident at once, so that the sweep keeps taking the CU slots that the frame's
// concurrent preprocessing and prior inference leave free.  512^3, 300-frame stream:
// 3072 blocks 4482-4494 frames/s and 54 us for the sweep alone, 6144 blocks 4489-4490 and
// 87 us, 1536 blocks 4374-4377 and 49 us.
constexpr int kSweepListBlocks = 3072;
constexpr uint32_t kSweepXcdChunk = 16;  // consecutive sweep blocks kept on one XCD
// x-slices of a brick whose loads a wavefront issues together: four (70 VGPRs for FP16, 72
// for FP32 voxels, seven waves per SIMD) beat all eight at once (98 VGPRs, five waves per
// SIMD).  A wave's first list entry loaded beside the counts takes FP32 to 74, six waves,
// and gave nothing.
constexpr int kSlicePass = 4;
constexpr uint8_t kBrickSkip = 0, kBrickFree = 1, kBrickExact = 2;
constexpr int kTileRow = 8;  // most raylen tiles in one row of a footprint (tile_range)
// Bricks whose classing waves (64 bricks each) the chip holds at once, three per SIMD: 1,024
// x 3 x 64.  Eight kf_integrate calls over four rooms, two rows a wait / one: 256^3 146-152 /
// 151-155 us, 384^3 149-170 / 152-170, 448^3 159-179 / 157-178, 480^3 168-195 / 165-188, 512^3
// 170-208 / 169-203, 768^3 291-385 / 289-387.
constexpr int kLatencyBricks = 196608;

struct SweepArgs {
  void* vox;
  uint32_t* count;  // [exact, free]: entries of each class in list
  uint32_t* list;   // bricks to visit: bx << 24 | by << 16 | bz << 8 | class; the exact ones
                    // from the front, the free ones from the back (list[cap - 1 - i])
  uint32_t cap;     // entries list holds (nb^3)
  int nb;           // bricks per axis
  float2* t8;       // raylen (min, max) per 8x8 tile, w8 per row
  float2* t32;      // per 32x32 tile, w32 per row
  int w8, w32;
  const float* raylen;
  const kf_pose* pose;
  unsigned long long* updated;
  uint32_t* mask;
  OccMap occ;  // brick occupancy map (occ.words NULL: none)
  int n;
  float h, ox, oy, oz;
  float fx, fy, cx, cy;
  int W, H;
  float dmin, dmax;
  float trunc, inv_trunc, maxw;
  float band;  // T + max(0.01 T, 0.1 mm): half-width of the band where the square root is taken
};

// One 16-byte store per thread, no loop (launch_items: more than 2^31 take several
// launches).  Bound by memory; 512 MB: 78 us, 6.8 TB/s (a grid-stride loop 117 us on 8192
// blocks, 96 on 16384; two or more stores a thread 88 and up), 128 MB: 20.6 us against 21.9.
__global__ __launch_bounds__(kItemThreads) void volume_fill(uint4* p, size_t n16, uint4 word) {
  const size_t i = (size_t)blockIdx.x * kItemThreads + threadIdx.x;
  if (i < n16) p[i] = word;
}

// Raylen extrema of the 8x8 and 32x32 pixel tiles (x = min, y = max).  Pixels
// outside the image are ignored; invalid pixels (raylen 0) count, so a tile with
// one has min 0.  One 256-thread block per 32x32 tile, a 2x2 quad per thread.
__global__ __launch_bounds__(256) void raylen_tiles(const float* rl, int W, int H, float2* t8, int w8,
                                                    float2* t32, int w32, uint32_t* list_count) {
  __shared__ float qmin[16][16], qmax[16][16], s8[2][16];
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < 2) list_count[threadIdx.x] = 0;  // the next kernel fills them
  const int qx = threadIdx.x & 15, qy = threadIdx.x >> 4;
  const int x0 = blockIdx.x * 32 + 2 * qx, y0 = blockIdx.y * 32 + 2 * qy;
  float mn = 3.0e38f, mx = 0.0f;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const int x = x0 + (d & 1), y = y0 + (d >> 1);
    if (x < W && y < H) {
      const float r = rl[y * W + x];
      mn = fminf(mn, r);
      mx = fmaxf(mx, r);
    }
  }
  qmin[qy][qx] = mn;
  qmax[qy][qx] = mx;
  __syncthreads();
  if (threadIdx.x < 16) {
    const int i = threadIdx.x & 3, j = threadIdx.x >> 2;  // 8x8 tile (i, j) of the 32x32 tile
    float a = 3.0e38f, b = 0.0f;
    for (int v = 0; v < 4; ++v)
      for (int u = 0; u < 4; ++u) {
        a = fminf(a, qmin[4 * j + v][4 * i + u]);
        b = fmaxf(b, qmax[4 * j + v][4 * i + u]);
      }
    s8[0][threadIdx.x] = a;
    s8[1][threadIdx.x] = b;
    const int tx = blockIdx.x * 4 + i, ty = blockIdx.y * 4 + j;
    if (tx * 8 < W && ty * 8 < H) t8[ty * w8 + tx] = make_float2(a, b);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    float a = 3.0e38f, b = 0.0f;
    for (int q = 0; q < 16; ++q) {
      a = fminf(a, s8[0][q]);
      b = fmaxf(b, s8[1][q]);
    }
    t32[blockIdx.y * w32 + blockIdx.x] = make_float2(a, b);
  }
}

// Raylen extrema over the pixels [u0, u1] x [v0, v1] (a superset: whole tiles), from
// the 8x8 tiles when the range is small, else the 32x32 ones; false when it is too
// large for either.
//
// A row of the range holds at most 6 (8x8) or 8 (32x32) tiles: its loads are issued
// together, one wait for them.  LATENCY: those of two rows, all lanes taking part (past the
// range: its last tile again); else a row's, lanes past their range taking no part.  Classing
// few bricks is a chain of latencies, where the first form is the faster; once the bricks'
// waves no longer fit the chip together its extra loads cost more (kLatencyBricks).
template <bool LATENCY>
__device__ __forceinline__ bool tile_range(const SweepArgs& a, int u0, int u1, int v0, int v1, float& mn,
                                           float& mx) {
  int sh;
  const float2* t;
  int w;
  if (u1 - u0 <= 40 && v1 - v0 <= 40) {
    sh = 3;
    t = a.t8;
    w = a.w8;
  } else if (u1 - u0 <= 200 && v1 - v0 <= 200) {
    sh = 5;
    t = a.t32;
    w = a.w32;
  } else {
    return false;
  }
  mn = 3.0e38f;
  mx = 0.0f;
  constexpr int ROWS = LATENCY ? 2 : 1;
  const int tx0 = u0 >> sh, tx1 = u1 >> sh, ty1 = v1 >> sh;
  for (int ty = v0 >> sh; ty <= ty1; ty += ROWS) {
    float2 e[ROWS][kTileRow];
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      const float2* row = t + min(ty + i, ty1) * w;
#pragma unroll
      for (int j = 0; j < kTileRow; ++j) {
        if constexpr (LATENCY)
          e[i][j] = row[min(tx0 + j, tx1)];
        else
          e[i][j] = tx0 + j <= tx1 ? row[tx0 + j] : make_float2(3.0e38f, 0.0f);
      }
    }
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
#pragma unroll
      for (int j = 0; j < kTileRow; ++j) {
        mn = fminf(mn, e[i][j].x);
        mx = fmaxf(mx, e[i][j].y);
      }
    }
  }
  return true;
}

// Sweep class of each 8^3 brick (one thread per brick).  The brick's voxel centres
// span the box of its eight corner centres; camera coordinates are affine in the
// voxel position, so depth and distance extremes lie at corners and the image of
// the box (all corners in front of the camera) is the convex hull of the corner
// images.  With the FP32 pose and grid that the per-voxel test uses, evaluated in
// FP64:
//   skip : all corners before min_depth or beyond max_depth, or the footprint
//          misses the updatable pixels (rounded u in [2, W-3], v in [2, H-3]), or
//          the nearest point of the box is farther than the largest raylen under
//          the footprint plus the band: no voxel is updated (the per-voxel test
//          rejects it on depth, image bounds, an invalid pixel or sdf < -T);
//   free : every corner inside the depth range, the footprint inside the
//          updatable pixels, every raylen under it valid, and the farthest corner
//          nearer than the smallest raylen minus the band: every voxel is updated
//          with f = 1 (the test's free-space shortcut);
//   exact: otherwise.
// Margins: 0.05 px, 1e-4 m in depth, 2e-4 m in distance, against FP32 errors of the
// per-voxel path below 4e-3 px and 2e-6 m.
template <bool LATENCY>
__device__ __forceinline__ uint8_t classify_brick(const SweepArgs& a, int bx, int by, int bz) {
  const kf_posef P = a.pose->cw;
  double R[9], t[3];
  for (int q = 0; q < 9; ++q) R[q] = (double)P.r[q];
  for (int q = 0; q < 3; ++q) t[q] = (double)P.t[q];
  const double h = (double)a.h;
  const double lo[3] = {(double)a.ox + (8.0 * bx + 0.5) * h, (double)a.oy + (8.0 * by + 0.5) * h,
                        (double)a.oz + (8.0 * bz + 0.5) * h};
  const double e7 = 7.0 * h;
  const double hi[3] = {lo[0] + e7, lo[1] + e7, lo[2] + e7};
  // Camera points of the corners: the lo corner plus the edge steps R e_k 7h
  // (additions in place of eight matrix products; FP64 rounding ~1e-16 m).
  double q[4][3];  // corners (x, y) = (0,0), (0,1), (1,0), (1,1) at z = lo
  for (int r = 0; r < 3; ++r) {
    q[0][r] = (R[3 * r] * lo[0] + R[3 * r + 1] * lo[1]) + R[3 * r + 2] * lo[2] + t[r];
    q[1][r] = q[0][r] + R[3 * r + 1] * e7;
    q[2][r] = q[0][r] + R[3 * r] * e7;
    q[3][r] = q[2][r] + R[3 * r + 1] * e7;
  }
  double pzmin = 1e300, pzmax = -1e300, umin = 1e300, umax = -1e300, vmin = 1e300, vmax = -1e300, d2max = 0.0;
  for (int c = 0; c < 8; ++c) {
    const double* b = q[c >> 1];
    const double px = (c & 1) ? b[0] + R[2] * e7 : b[0];
    const double py = (c & 1) ? b[1] + R[5] * e7 : b[1];
    const double pz = (c & 1) ? b[2] + R[8] * e7 : b[2];
    pzmin = fmin(pzmin, pz);
    pzmax = fmax(pzmax, pz);
    d2max = fmax(d2max, fma(px, px, fma(py, py, pz * pz)));
    // The image bounds are used only when every corner has pz > 1e-3, so they are
    // formed unconditionally.  1 / pz: the hardware reciprocal refined by two
    // Newton steps (relative error ~1e-16, far inside the 0.05 px margin).
    double iz = __builtin_amdgcn_rcp(pz);
    iz = fma(iz, fma(-pz, iz, 1.0), iz);
    iz = fma(iz, fma(-pz, iz, 1.0), iz);
    const double u = fma((double)a.fx * px, iz, (double)a.cx), v = fma((double)a.fy * py, iz, (double)a.cy);
    umin = fmin(umin, u);
    umax = fmax(umax, u);
    vmin = fmin(vmin, v);
    vmax = fmax(vmax, v);
  }
  const double mz = 1e-4, md = 2e-4, mpx = 0.05;
  uint8_t cls = kBrickExact;
  if (pzmax < (double)a.dmin - mz || pzmin > (double)a.dmax + mz) {
    cls = kBrickSkip;
  } else if (pzmin > 1e-3) {
    umin -= mpx;
    umax += mpx;
    vmin -= mpx;
    vmax += mpx;
    const double ulo = 1.5, uhi = (double)a.W - 2.5, vlo = 1.5, vhi = (double)a.H - 2.5;
    if (umax < ulo || umin >= uhi || vmax < vlo || vmin >= vhi) {
      cls = kBrickSkip;
    } else {
      const int pu0 = (int)fmax(2.0, floor(umin + 0.5)), pu1 = (int)fmin((double)(a.W - 3), floor(umax + 0.5));
      const int pv0 = (int)fmax(2.0, floor(vmin + 0.5)), pv1 = (int)fmin((double)(a.H - 3), floor(vmax + 0.5));
      float rmin, rmax;
      if (pu0 <= pu1 && pv0 <= pv1 && tile_range<LATENCY>(a, pu0, pu1, pv0, pv1, rmin, rmax)) {
        const bool inside = umin >= ulo && umax < uhi && vmin >= vlo && vmax < vhi;
        // nearest point of the box to the camera centre -R^T t
        double dn2 = 0.0;
        for (int k = 0; k < 3; ++k) {
          const double ck = -(R[k] * t[0] + R[3 + k] * t[1] + R[6 + k] * t[2]);
          const double e = ck < lo[k] ? lo[k] - ck : (ck > hi[k] ? ck - hi[k] : 0.0);
          dn2 += e * e;
        }
        const double band = (double)a.band;
        if (inside && pzmin >= (double)a.dmin + mz && pzmax <= (double)a.dmax - mz && rmin > 0.0f &&
            sqrt(d2max) + md < (double)rmin - band)
          cls = kBrickFree;
        else if (sqrt(dn2) - md > (double)rmax + band)
          cls = kBrickSkip;
      }
    }
  }
  return cls;
}

// One thread per brick; exact bricks are appended to the front of the work list and
// free ones to its back (one atomic per block and class; entries in brick order
// within a block), so that the sweep can deal each wavefront its share of both.
template <bool LATENCY>
__global__ __launch_bounds__(256) void brick_classify(SweepArgs a) {
  __shared__ uint32_t s_cnt[2][4], s_base[2];
  const int nb = a.nb;
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  const int bx = b / (nb * nb), r = b - bx * (nb * nb), by = r / nb, bz = r - by * nb;
  const uint8_t cls = b < nb * nb * nb ? classify_brick<LATENCY>(a, bx, by, bz) : kBrickSkip;
  const int c = cls == kBrickExact ? 0 : 1;  // list part: 0 exact, 1 free
  const unsigned long long m[2] = {__ballot(cls == kBrickExact), __ballot(cls == kBrickFree)};
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & (kWave - 1);
  if (lane < 2) s_cnt[lane][wave] = (uint32_t)__popcll(m[lane]);
  __syncthreads();
  if (threadIdx.x < 2) {
    const int q = threadIdx.x;
    const uint32_t tot = (s_cnt[q][0] + s_cnt[q][1]) + (s_cnt[q][2] + s_cnt[q][3]);
    s_base[q] = tot ? atomicAdd(a.count + q, tot) : 0u;
  }
  __syncthreads();
  if (cls != kBrickSkip) {
    uint32_t off = s_base[c] + (uint32_t)__popcll(m[c] & ((1ull << lane) - 1ull));
    for (int w = 0; w < wave; ++w) off += s_cnt[c][w];
    a.list[c == 0 ? off : a.cap - 1u - off] =
        ((uint32_t)bx << 24) | ((uint32_t)by << 16) | ((uint32_t)bz << 8) | cls;
  }
}

// Exact per-voxel test in two parts, so that a wave can issue the raylen loads of
// several chunks before using any.  voxel_project: camera point of voxel z of the
// column, depth gate, projection with round half up and image bounds; returns the
// pixel index (-1: not updated) and d2 = |p|^2.  voxel_finish: the test at that
// pixel; true and the new normalised sample f if updated.
struct VoxProj {
  float d2;
  int pix;
};

__device__ __forceinline__ VoxProj voxel_project(const SweepArgs& a, float ax, float ay, float az, const float* r,
                                                 int k) {
  VoxProj q;
  q.pix = -1;
  q.d2 = 0.0f;
  const float wz = a.oz + ((float)k + 0.5f) * a.h;
  const float px = ax + r[2] * wz;
  const float py = ay + r[5] * wz;
  const float pz = az + r[8] * wz;
  if (!(pz >= a.dmin && pz <= a.dmax)) return q;
  const float iz = 1.0f / pz;
  const float u = (a.fx * px + a.cx * pz) * iz;
  const float v = (a.fy * py + a.cy * pz) * iz;
  const float ru = round_half_up(u);
  const float rv = round_half_up(v);
  if (!(ru >= 2.0f && ru < (float)(a.W - 2) && rv >= 2.0f && rv < (float)(a.H - 2))) return q;
  q.pix = (int)rv * a.W + (int)ru;
  q.d2 = (px * px + py * py) + pz * pz;
  return q;
}

__device__ __forceinline__ bool voxel_finish(const SweepArgs& a, float rl, float d2, float& f) {
  if (!(rl > 0.0f)) return false;
  // Outside |rl - dist| <= band the outcome follows from d2 alone: the margin
  // band - T >= max(0.01 T, 0.1 mm) is far above the FP32 error of d2, lo^2, hi^2,
  // dist and sdf (< 2 um for rays up to 10 m), so free space yields exactly f = 1
  // (sdf / T > 1 clamps to 1) and the far side is exactly "not updated" (sdf < -T),
  // as the full expression gives.
  const float lo = rl - a.band, hi = rl + a.band;
  if (lo > 0.0f && d2 < lo * lo) {
    f = 1.0f;
    return true;
  }
  if (d2 > hi * hi) return false;
  const float dist = sqrtf(d2);
  const float sdf = rl - dist;
  if (sdf < -a.trunc) return false;
  f = fmaxf(fminf(sdf * a.inv_trunc, 1.0f), -1.0f);
  return true;
}

// Marks brick (bx, by, bz) in the occupancy map (only when the bit is missing).
__device__ __forceinline__ void occ_mark_brick(const OccMap& occ, int bx, int by, int bz) {
  unsigned long long* w = occ.words + ((bx * occ.nb + by) * occ.per_col + (bz >> 6));
  const unsigned long long bit = 1ull << (bz & 63);
  if (__hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & bit) return;
  __hip_atomic_fetch_or(w, bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The sweep over the listed bricks.  Lane (yy, zz) = (lane >> 3, lane & 7) holds
// voxel (8 bx + xs, 8 by + yy, 8 bz + zz) of each x-slice xs; the eight slices'
// loads (and, for exact bricks, their raylen loads) are issued together.
template <int FMT>
__global__ __launch_bounds__(256) void integrate(SweepArgs a) {
  using Word = typename std::conditional<FMT == KF_VOXEL_F16, uint32_t, float2>::type;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
  const int yy = lane >> 3, zz = lane & 7;
  const kf_posef P = a.pose->cw;
  // entry k: the k-th exact brick, then the free ones; waves stride over k, so each
  // takes an even share of each class
  const size_t n = (size_t)a.n, slice = n * n;
  int count = 0;
  // Blocks reach the 8 XCDs (each with its own L2) round-robin.  Consecutive list
  // entries are mostly z-neighbouring bricks, whose 32-byte voxel rows share 128-byte
  // lines, so chunks of kSweepXcdChunk consecutive blocks are remapped onto one XCD
  // (one L2 fetches the lines once) while the chunks still rotate over the XCDs
  // (the clustered exact bricks stay spread): 132 -> 85 MB read per sweep at 512^3.
  const uint32_t G = gridDim.x;
  uint32_t lb = blockIdx.x;
  if (G % (8u * kSweepXcdChunk) == 0u) {
    const uint32_t x = blockIdx.x % 8u, j = blockIdx.x / 8u;
    lb = ((j / kSweepXcdChunk) * 8u + x) * kSweepXcdChunk + j % kSweepXcdChunk;
  }
  const uint32_t n_exact = a.count[0], items = n_exact + a.count[1];
  for (uint32_t i = lb * kWavesPerBlock + wave; i < items; i += G * kWavesPerBlock) {
    const uint32_t e = a.list[i < n_exact ? i : a.cap - 1u - (i - n_exact)];
    const int bx = (int)(e >> 24), by = (int)((e >> 16) & 255u), bz = (int)((e >> 8) & 255u);
    const bool exact = (e & 255u) == kBrickExact;  // uniform
    const int y = 8 * by + yy, z = 8 * bz + zz;
    Word* base = static_cast<Word*>(a.vox) + ((size_t)(8 * bx) * n + (size_t)y) * n + (size_t)z;
    bool nz_any = false, nz_x0 = false;  // f != 1 written: anywhere / in slice 0
#pragma unroll
    for (int x0 = 0; x0 < 8; x0 += kSlicePass) {
      bool upd[kSlicePass];
      float fs[kSlicePass], rl[kSlicePass];
      VoxProj q[kSlicePass];
#pragma unroll
      for (int j = 0; j < kSlicePass; ++j) {
        fs[j] = 1.0f;
        q[j].pix = -1;
        q[j].d2 = 0.0f;
      }
      if (exact) {
        const float wy = a.oy + ((float)y + 0.5f) * a.h;
#pragma unroll
        for (int j = 0; j < kSlicePass; ++j) {
          const float wx = a.ox + ((float)(8 * bx + x0 + j) + 0.5f) * a.h;
          const float ax = (P.r[0] * wx + P.r[1] * wy) + P.t[0];
          const float ay = (P.r[3] * wx + P.r[4] * wy) + P.t[1];
          const float az = (P.r[6] * wx + P.r[7] * wy) + P.t[2];
          q[j] = voxel_project(a, ax, ay, az, P.r, z);
        }
      }
      // one batch of loads (no branches: lanes without a pixel read pixel 0 and ignore it)
      Word wv[kSlicePass];
#pragma unroll
      for (int j = 0; j < kSlicePass; ++j) {
        rl[j] = a.raylen[q[j].pix >= 0 ? q[j].pix : 0];
        wv[j] = base[(x0 + j) * slice];
      }
#pragma unroll
      for (int j = 0; j < kSlicePass; ++j) {
        const int xs = x0 + j;
        upd[j] = !exact || (q[j].pix >= 0 && voxel_finish(a, rl[j], q[j].d2, fs[j]));
        if (!upd[j]) continue;
        ++count;
        bool nz;
        if (FMT == KF_VOXEL_F16) {
          const uint32_t w = reinterpret_cast<const uint32_t&>(wv[j]);
          const float fo = half_bits_to_float(w & 0xffffu);
          const float wo = (float)(w >> 16);
          // Free space (f_old = f = 1) averages to exactly 1: (w + 1) / (w + 1).
          const float fn = (fo == 1.0f && fs[j] == 1.0f) ? 1.0f : (fo * wo + fs[j]) / (wo + 1.0f);
          const float wn = fminf(wo + 1.0f, a.maxw);
          const uint32_t nw = float_to_half_bits(fn) | ((uint32_t)wn << 16);
          // saturated free space (f = 1, w = max) is left as it is
          if (nw != w) reinterpret_cast<uint32_t*>(base)[xs * slice] = nw;
          nz = (nw & 0xffffu) != 0x3C00u;
        } else {
          const float2 v = reinterpret_cast<const float2&>(wv[j]);
          const float fn = (v.x == 1.0f && fs[j] == 1.0f) ? 1.0f : (v.x * v.y + fs[j]) / (v.y + 1.0f);
          const float wn = fminf(v.y + 1.0f, a.maxw);
          if (__float_as_uint(fn) != __float_as_uint(v.x) || __float_as_uint(wn) != __float_as_uint(v.y))
            reinterpret_cast<float2*>(base)[xs * slice] = make_float2(fn, wn);
          nz = fn != 1.0f;
        }
        nz_any = nz_any || nz;
        if (xs == 0) nz_x0 = nz;
      }
      if (a.mask) {  // per slice: eight rows of eight z-bits, each inside one 32-bit word
#pragma unroll
        for (int j = 0; j < kSlicePass; ++j) {
          const unsigned long long m = __ballot(upd[j]);
          const uint32_t bits = (uint32_t)(m >> (8 * yy)) & 0xffu;
          if (zz == 0 && bits) {
            const size_t v0 = ((size_t)(8 * bx + x0 + j) * n + (size_t)y) * n + (size_t)(8 * bz);
            atomicOr(&a.mask[v0 >> 5], bits << (v0 & 31));
          }
        }
      }
    }
    if (a.occ.words) {
      // A clear brick bit promises f == 1 on the brick extended by one voxel along +x,
      // +y, +z: a voxel with f != 1 marks its brick and, on the low face of an axis,
      // the neighbour below along that axis.
      const unsigned long long A = __ballot(nz_any), X = __ballot(nz_x0);
      if (A) {  // uniform
        const unsigned long long Y0 = 0xffull, Z0 = 0x0101010101010101ull;  // lanes yy == 0 / zz == 0
        if (lane < 8) {
          const int dx = lane & 1, dy = (lane >> 1) & 1, dz = lane >> 2;
          const unsigned long long src = (dx ? X : A) & (dy ? Y0 : ~0ull) & (dz ? Z0 : ~0ull);
          if (src && bx >= dx && by >= dy && bz >= dz) occ_mark_brick(a.occ, bx - dx, by - dy, bz - dz);
        }
      }
    }
  }
  if (a.updated) {  // one device atomic per block (uniform branch)
    __shared__ int red[kWavesPerBlock];
    count = wave_sum_i_lane63(count);
    if (lane == 63) red[wave] = count;
    __syncthreads();
    if (threadIdx.x == 0) {
      const int tot = (red[0] + red[1]) + (red[2] + red[3]);
      if (tot) atomicAdd(a.updated, (unsigned long long)tot);
    }
  }
}

// Whole-volume occupancy statistics: one pass over every voxel with 16-byte
// loads, block reduction in LDS, one FP64 atomic per block and statistic.
template <int FMT>
__global__ __launch_bounds__(256) void volume_stats(const uint4* p, size_t n16, double* out) {
  double obs = 0.0, sw = 0.0, sf = 0.0, neg = 0.0;
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < n16; i += stride) {
    const uint4 q = p[i];
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
    if (FMT == KF_VOXEL_F16) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float wt = (float)(w[j] >> 16);
        if (wt > 0.0f) {
          const float f = half_bits_to_float(w[j] & 0xffffu);
          obs += 1.0;
          sw += wt;
          sf += f;
          neg += f < 0.0f ? 1.0 : 0.0;
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const float f = __uint_as_float(w[2 * j]), wt = __uint_as_float(w[2 * j + 1]);
        if (wt > 0.0f) {
          obs += 1.0;
          sw += wt;
          sf += f;
          neg += f < 0.0f ? 1.0 : 0.0;
        }
      }
    }
  }
  __shared__ double red[4][256];
  red[0][threadIdx.x] = obs;
  red[1][threadIdx.x] = sw;
  red[2][threadIdx.x] = sf;
  red[3][threadIdx.x] = neg;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o)
      for (int q = 0; q < 4; ++q) red[q][threadIdx.x] += red[q][threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x < 4) atomicAdd(&out[threadIdx.x], red[threadIdx.x][0]);
}

// Occupancy from scratch: one wavefront per (voxel column, occupancy word) task,
// waves striding over the tasks.  Word kw holds bricks 64 kw .. 64 kw + 63, whose
// extended extents cover voxels z in [512 kw, 512 kw + 512] (the last one also
// belongs to the next word's first brick); the wave reads them with 16-byte loads
// and marks the bricks that hold f != 1.
__device__ __forceinline__ unsigned long long occ_zbits_word(int z, int kw) {
  const int b = (z >> 3) - kOccWordBricks * kw;  // brick of z relative to the word
  unsigned long long m = (b >= 0 && b < kOccWordBricks) ? 1ull << b : 0ull;
  if ((z & 7) == 0 && b >= 1 && b <= kOccWordBricks) m |= 1ull << (b - 1);
  return m;
}

template <int FMT>
__global__ __launch_bounds__(256) void occupancy_rebuild(const void* vox, int n, OccMap occ) {
  constexpr int V = (FMT == KF_VOXEL_F16) ? 4 : 2;  // voxels per 16-byte load
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
  const int tasks = n * n * occ.per_col;
  for (int c = blockIdx.x * kWavesPerBlock + wave; c < tasks; c += gridDim.x * kWavesPerBlock) {
    const int colno = c / occ.per_col, kw = c - colno * occ.per_col;
    const int ix = colno / n, iy = colno - ix * n;
    const size_t col = (size_t)colno * (size_t)n;
    const int z0 = kw * kOccWordBricks * 8, z1 = min(n, z0 + kOccWordBricks * 8 + 1);  // voxels [z0, z1)
    unsigned long long bits = 0ull;
    // zb is a multiple of V and below z1 <= n (a multiple of 8): the load stays in the column
    for (int zb = z0 + lane * V; zb < z1; zb += kWave * V) {
      const uint4 q = *reinterpret_cast<const uint4*>(static_cast<const uint32_t*>(vox) + (FMT == KF_VOXEL_F16 ? col + zb : 2 * (col + zb)));
      if (FMT == KF_VOXEL_F16) {
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (zb + j < z1 && (w[j] & 0xffffu) != 0x3C00u) bits |= occ_zbits_word(zb + j, kw);
      } else {
        if (__uint_as_float(q.x) != 1.0f) bits |= occ_zbits_word(zb, kw);
        if (zb + 1 < z1 && __uint_as_float(q.z) != 1.0f) bits |= occ_zbits_word(zb + 1, kw);
      }
    }
    occ_mark_column(occ, ix, iy, kw, bits, lane);
  }
}

// Brick distances, min(Chebyshev distance in bricks to the nearest set brick,
// kBrickDistCap).  The distance of brick (x, y, z) is the number of radii r in
// 0..cap-1 for which the cube of radius r around it holds no set brick; the cube's
// set bricks are the bits of the OR over the (2r+1)^2 columns around (x, y) (bit bz
// of column word (bx, by)), dilated by r along the word.  The square-window ORs come
// from a sparse table in LDS: T_k(x, y) = OR over the 2^k x 2^k columns from (x, y),
// built for k = 1..4 by doubling, and a window of side L is the OR of four T_k with
// 2^k <= L < 2^(k+1).  One block per 8 x 8 tile of columns stages the tile plus a
// halo of cap - 1 columns (out-of-volume columns empty) and builds the table; then
// its sixteen wavefronts test one radius each for the tile's 64 columns (lane t:
// column (x0 + t % 8, y0 + t / 8)), and the first forms each column's 64 distances
// in five bit planes and writes them as one 64-byte row.
constexpr int kDistTile = 8;
constexpr int kDistHalo = kBrickDistCap - 1;
constexpr int kDistSide = kDistTile + 2 * kDistHalo;
constexpr int kDistLevels = 5;  // T_0 .. T_4: windows up to 2 * 15 + 1 = 31 < 32 columns
constexpr int kDistThreads = 1024;  // sixteen wavefronts: one radius each, two table cells per thread and level
constexpr int kRadiiPerWave = kBrickDistCap / (kDistThreads / kWave);  // radii each wavefront tests
static_assert(2 * kDistHalo + 1 < (1 << kDistLevels), "window wider than the largest table level");
static_assert(kRadiiPerWave * (kDistThreads / kWave) == kBrickDistCap && kBrickDistCap == 16,
              "the count planes below assume 16 radii split evenly over the wavefronts");

// OR of w shifted by -r .. r bits (bits leaving the word are bricks outside the volume)
__device__ __forceinline__ unsigned long long dilate_bits(unsigned long long w, int r) {
  unsigned long long up = w, down = w;
  int len = 1;
  while (2 * len <= r + 1) {
    up |= up << len;
    down |= down >> len;
    len *= 2;
  }
  const int rest = r + 1 - len;  // up = OR over shifts 0 .. len-1; extend to 0 .. r
  up |= up << rest;
  down |= down >> rest;
  return up | down;
}

// Columns of more than 64 bricks (per_col > 1 words) are processed in chunks of 32
// output bricks, blockIdx.z = chunk c: the chunk word holds bricks 32c - 16 ..
// 32c + 47 (bits outside the volume clear), and the counts of its bits 16 .. 47 —
// bricks 32c .. 32c + 31 — only involve dilations by at most 15 bits that stay
// inside the word.  With one word per column the word is the whole column.
__device__ __forceinline__ int dist_chunk_first_brick(const OccMap& occ, int c) {
  return occ.per_col == 1 ? 0 : 32 * c - 16;
}

// Bits s .. s + 63 of brick column `col` (bits outside 0 .. 64 per_col - 1 read 0).
__device__ __forceinline__ unsigned long long column_bits(const OccMap& occ, int col, int s) {
  const int w = s >> 6, sh = s & 63;  // arithmetic shift: w = floor(s / 64)
  const unsigned long long* cw = occ.words + (size_t)col * occ.per_col;
  const unsigned long long lo = (w >= 0 && w < occ.per_col) ? cw[w] : 0ull;
  if (sh == 0) return lo;
  const unsigned long long hi = (w + 1 >= 0 && w + 1 < occ.per_col) ? cw[w + 1] : 0ull;
  return (lo >> sh) | (hi << (64 - sh));
}

__global__ __launch_bounds__(kDistThreads) void brick_distance(OccMap occ, uint8_t* out) {
  __shared__ unsigned long long t[kDistLevels][kDistSide * kDistSide];
  constexpr int kCells = kDistSide * kDistSide;
  constexpr int kPer = (kCells + kDistThreads - 1) / kDistThreads;  // cells per thread and level
  const int nb = occ.nb, tid = threadIdx.x;
  const int x0 = blockIdx.x * kDistTile - kDistHalo, y0 = blockIdx.y * kDistTile - kDistHalo;
  const int s0 = dist_chunk_first_brick(occ, blockIdx.z);
  {
    // every load in flight at once: out-of-range cells read a clamped column and drop it
    unsigned long long v[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int i = tid + j * kDistThreads;
      const int x = x0 + i / kDistSide, y = y0 + i % kDistSide;
      const bool in = i < kCells && x >= 0 && x < nb && y >= 0 && y < nb;
      const int xc = min(max(x, 0), nb - 1), yc = min(max(y, 0), nb - 1);
      const unsigned long long w = column_bits(occ, xc * nb + yc, s0);
      v[j] = in ? w : 0ull;
    }
#pragma unroll
    for (int j = 0; j < kPer; ++j)
      if (tid + j * kDistThreads < kCells) t[0][tid + j * kDistThreads] = v[j];
  }
  __syncthreads();
#pragma unroll
  for (int k = 1; k < kDistLevels; ++k) {
    // T_k(a, b) for a, b + 2^k <= side from four T_(k-1) of half the side; all reads
    // of a level before its writes (cells past the end recompute the last one)
    const int h = 1 << (k - 1), n = kDistSide - (1 << k) + 1;
    unsigned long long v[kPer];
    int at[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int i = min(tid + j * kDistThreads, n * n - 1);
      at[j] = (i / n) * kDistSide + i % n;
      const unsigned long long* p = &t[k - 1][at[j]];
      v[j] = p[0] | p[h] | p[h * kDistSide] | p[h * kDistSide + h];
    }
#pragma unroll
    for (int j = 0; j < kPer; ++j)
      if (tid + j * kDistThreads < n * n) t[k][at[j]] = v[j];
    __syncthreads();
  }
  // Lane t of each wavefront owns column (x0 + t % 8, y0 + t / 8); wavefront q finds,
  // for radii r = kRadiiPerWave q .. + kRadiiPerWave - 1, the mask e_r of the column's
  // bricks whose cube of radius r holds no set brick.
  __shared__ unsigned long long em[kBrickDistCap][kWave];
  const int wave = tid >> 6, lane = tid & (kWave - 1);
  const int tx = lane % kDistTile, ty = lane / kDistTile;
  const int lx = kDistHalo + tx, ly = kDistHalo + ty;
#pragma unroll
  for (int q = 0; q < kRadiiPerWave; ++q) {
    const int r = kRadiiPerWave * wave + q;
    const int k = 31 - __builtin_clz(2 * r + 1), side = 1 << k;
    const int a = lx - r, b = lx + r + 1 - side, c = ly - r, d = ly + r + 1 - side;
    const unsigned long long* T = t[k];
    const unsigned long long w = T[a * kDistSide + c] | T[b * kDistSide + c] | T[a * kDistSide + d] |
                                 T[b * kDistSide + d];
    em[r][lane] = ~dilate_bits(w, r);
  }
  __syncthreads();
  if (wave != 0) return;  // one wavefront writes the tile's distances
  const int ox = blockIdx.x * kDistTile + tx, oy = blockIdx.y * kDistTile + ty;
  if (ox >= nb || oy >= nb) return;
  // The cube of radius r holds the one of radius r - 1, so the masks are nested
  // (e_r within e_(r-1)) and a brick's distance min(d, cap) is the number of radii r
  // whose e_r holds it: d >= j exactly when e_(j-1) does.  Its binary digits: the 16s
  // are e_15, the 8s e_7 outside e_15, the 4s e_3 outside e_7 or e_11 outside e_15,
  // and so on down to the 1s: e_(2i) outside e_(2i+1).
  unsigned long long e[kBrickDistCap];
#pragma unroll
  for (int r = 0; r < kBrickDistCap; ++r) e[r] = em[r][lane];
  unsigned long long cnt[5] = {0ull, 0ull, 0ull, 0ull, e[15]};  // bit planes of the counts
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int step = 1 << q;  // plane q: e_(m - 1) outside e_(m - 1 + step), m = step, 3 step, 5 step, ...
#pragma unroll
    for (int m = step; m < kBrickDistCap; m += 2 * step) cnt[q] |= e[m - 1] & ~e[m - 1 + step];
  }
  // byte b of the chunk = count of chunk bit b; 4 bricks per dword, bit j of a nibble
  // spread to bit 8j by a multiply
  uint32_t dw[16];
#pragma unroll
  for (int g = 0; g < 16; ++g) {
    uint32_t v = 0;
#pragma unroll
    for (int q = 0; q < 5; ++q) {
      const uint32_t nib = (uint32_t)(cnt[q] >> (4 * g)) & 0xFu;
      v |= ((nib * 0x00204081u) & 0x01010101u) << q;
    }
    dw[g] = v;
  }
  // the row of the column (64 bytes per occupancy word); one word: all 64 bricks,
  // else bricks 32c .. 32c + 31 (chunk bits 16 .. 47, dwords 4 .. 11)
  uint8_t* row = out + ((size_t)ox * nb + oy) * (kOccWordBricks * occ.per_col);
  if (occ.per_col == 1) {
    uint4* r = reinterpret_cast<uint4*>(row);
#pragma unroll
    for (int g = 0; g < 4; ++g) r[g] = make_uint4(dw[4 * g], dw[4 * g + 1], dw[4 * g + 2], dw[4 * g + 3]);
  } else {
    uint4* r = reinterpret_cast<uint4*>(row + 32 * blockIdx.z);
    r[0] = make_uint4(dw[4], dw[5], dw[6], dw[7]);
    r[1] = make_uint4(dw[8], dw[9], dw[10], dw[11]);
  }
}

__global__ __launch_bounds__(256) void fill_u64(unsigned long long* p, int count, unsigned long long v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) p[i] = v;
}

__global__ void zero_doubles(double* p, int n) {
  if ((int)threadIdx.x < n) p[threadIdx.x] = 0.0;
}

}  // namespace

kf_status launch_volume_stats(const kf_volume* v, double* d_out, hipStream_t s) {
  KF_CHECK_ARG(d_out != nullptr, "out is NULL");
  hipLaunchKernelGGL(zero_doubles, dim3(1), dim3(64), 0, s, d_out, 4);
  KF_TRY(check_launch("zero_doubles"));
  const size_t n16 = v->bytes / 16;
  const int blocks = (int)std::min<size_t>((n16 + 255) / 256, 4096);
  if (v->desc.format == KF_VOXEL_F16)
    hipLaunchKernelGGL(volume_stats<KF_VOXEL_F16>, dim3(blocks), dim3(256), 0, s,
                       static_cast<const uint4*>(v->d_voxels), n16, d_out);
  else
    hipLaunchKernelGGL(volume_stats<KF_VOXEL_F32>, dim3(blocks), dim3(256), 0, s,
                       static_cast<const uint4*>(v->d_voxels), n16, d_out);
  return check_launch("volume_stats");
}

// The volume's occupancy map as the kernels take it (words NULL: no map, or the
// free-space skip is switched off).
OccMap occ_map(const kf_volume* v) {
  return OccMap{v->occ_enabled ? v->d_occ : nullptr, v->occ_nb, v->occ_words};
}

// The map to zero (a fill kernel, so that graph capture stays valid).
kf_status clear_occupancy(const kf_volume* v, hipStream_t s) {
  const int words = v->occ_nb * v->occ_nb * v->occ_words;
  hipLaunchKernelGGL(fill_u64, dim3(div_up(words, 256)), dim3(256), 0, s, v->d_occ, words, 0ull);
  return check_launch("fill_u64(occupancy)");
}

kf_status launch_volume_reset(kf_volume* v, hipStream_t s) {
  uint4 word;
  if (v->desc.format == KF_VOXEL_F16) {
    const uint32_t w = 0x3C00u;  // half(1.0), weight 0
    word = make_uint4(w, w, w, w);
  } else {
    const uint32_t one = 0x3F800000u;  // 1.0f, weight 0.0f
    word = make_uint4(one, 0u, one, 0u);
  }
  KF_TRY(launch_items(v->bytes / 16, [&](size_t first, size_t count, unsigned blocks) {
    hipLaunchKernelGGL(volume_fill, dim3(blocks), dim3(kItemThreads), 0, s, static_cast<uint4*>(v->d_voxels) + first, count,
                       word);
    return check_launch("volume_fill");
  }));
  if (v->d_occ) KF_TRY(clear_occupancy(v, s));  // every voxel is free space: all bricks clear
  v->occ_stale = false;
  return KF_OK;
}

kf_status launch_brick_distance(const kf_volume* v, hipStream_t s) {
  const OccMap occ = occ_map(v);
  if (!occ.words) return KF_OK;
  const int tiles = div_up(occ.nb, kDistTile);
  const int chunks = occ.per_col == 1 ? 1 : div_up(occ.nb, 32);
  hipLaunchKernelGGL(brick_distance, dim3(tiles, tiles, chunks), dim3(kDistThreads), 0, s, occ, v->d_bdist);
  return check_launch("brick_distance");
}

kf_status ensure_occupancy(const kf_volume* v, hipStream_t s) {
  const OccMap occ = occ_map(v);
  if (!occ.words || !v->occ_stale) return KF_OK;
  KF_TRY(clear_occupancy(v, s));
  const int n = v->desc.n;
  const int blocks = std::min(div_up(n * n * occ.per_col, kWavesPerBlock), kSweepMaxBlocks);
  if (v->desc.format == KF_VOXEL_F16)
    hipLaunchKernelGGL(occupancy_rebuild<KF_VOXEL_F16>, dim3(blocks), dim3(256), 0, s,
                       (const void*)v->d_voxels, n, occ);
  else
    hipLaunchKernelGGL(occupancy_rebuild<KF_VOXEL_F32>, dim3(blocks), dim3(256), 0, s,
                       (const void*)v->d_voxels, n, occ);
  KF_TRY(check_launch("occupancy_rebuild"));
  v->occ_stale = false;
  return KF_OK;
}

size_t sweep_tiles_floats2(const kf_intrinsics& k0) {
  return (size_t)div_up(k0.width, 8) * div_up(k0.height, 8) + (size_t)div_up(k0.width, 32) * div_up(k0.height, 32);
}

kf_status launch_raylen_tiles(const kf_intrinsics& k0, const float* d_raylen, const SweepTiles& t, hipStream_t s) {
  KF_CHECK_ARG(d_raylen && t.tiles && t.count, "raylen / tiles / count is NULL");
  KF_CHECK_ARG(k0.width <= kMaxImage && k0.height <= kMaxImage, "image too large");
  const int w8 = div_up(k0.width, 8), w32 = div_up(k0.width, 32);
  hipLaunchKernelGGL(raylen_tiles, dim3(w32, div_up(k0.height, 32)), dim3(256), 0, s, d_raylen, k0.width, k0.height,
                     t.tiles, w8, t.tiles + (size_t)w8 * div_up(k0.height, 8), w32, t.count);
  return check_launch("raylen_tiles");
}

kf_status launch_integrate(kf_volume* v, const kf_intrinsics& k0, const kf_integrate_params& p,
                           const float* d_raylen, const kf_pose* d_pose, unsigned long long* d_updated,
                           uint32_t* d_mask, hipStream_t s, hipEvent_t between, hipEvent_t kernel_start,
                           hipEvent_t kernel_stop, const SweepTiles* pre) {
  KF_CHECK_ARG(d_raylen && d_pose, "raylen/pose is NULL");
  KF_CHECK_ARG(p.min_depth_m >= 0.001f && p.max_depth_m > p.min_depth_m, "bad depth range");
  KF_CHECK_ARG(k0.width > 4 && k0.height > 4, "image too small");
  SweepArgs a;
  const kf_volume_desc& d = v->desc;
  a.vox = v->d_voxels;
  a.count = v->d_bricks;
  a.list = v->d_bricks + 2;
  a.nb = d.n / 8;
  a.cap = (uint32_t)a.nb * (uint32_t)a.nb * (uint32_t)a.nb;
  a.w8 = div_up(k0.width, 8);
  a.w32 = div_up(k0.width, 32);
  if (pre) {
    a.t8 = pre->tiles;
    a.t32 = pre->tiles + (size_t)a.w8 * div_up(k0.height, 8);
    a.count = pre->count;
  } else {
    a.t8 = v->d_rtiles;
    a.t32 = v->d_rtiles + kRayTiles8;
  }
  a.raylen = d_raylen;
  a.pose = d_pose;
  a.updated = d_updated;
  a.mask = d_mask;
  a.occ = occ_map(v);
  a.n = d.n;
  a.h = d.extent_m / (float)d.n;
  a.ox = d.origin_m[0];
  a.oy = d.origin_m[1];
  a.oz = d.origin_m[2];
  a.fx = k0.fx;
  a.fy = k0.fy;
  a.cx = k0.cx;
  a.cy = k0.cy;
  a.W = k0.width;
  a.H = k0.height;
  a.dmin = p.min_depth_m;
  a.dmax = p.max_depth_m;
  a.trunc = d.trunc_m;
  a.inv_trunc = 1.0f / d.trunc_m;
  a.band = d.trunc_m + std::max(0.01f * d.trunc_m, 1e-4f);
  a.maxw = d.max_weight;
  KF_CHECK_ARG(k0.width <= kMaxImage && k0.height <= kMaxImage, "image too large");
  if (!pre) {
    hipLaunchKernelGGL(raylen_tiles, dim3(div_up(k0.width, 32), div_up(k0.height, 32)), dim3(256), 0, s, d_raylen,
                       k0.width, k0.height, a.t8, a.w8, a.t32, a.w32, a.count);
    KF_TRY(check_launch("raylen_tiles"));
  }
  const int nbricks = a.nb * a.nb * a.nb;
  auto classify = nbricks <= kLatencyBricks ? brick_classify<true> : brick_classify<false>;
  hipLaunchKernelGGL(classify, dim3(div_up(nbricks, 256)), dim3(256), 0, s, a);
  KF_TRY(check_launch("brick_classify"));
  if (between) KF_HIP(hipEventRecord(between, s));
  const int blocks = std::min(div_up(nbricks, kWavesPerBlock), kSweepListBlocks);
  auto kern = d.format == KF_VOXEL_F16 ? integrate<KF_VOXEL_F16> : integrate<KF_VOXEL_F32>;
  if (kernel_start && kernel_stop)
    hipExtLaunchKernelGGL(kern, dim3(blocks), dim3(256), 0, s, kernel_start, kernel_stop, 0, a);
  else
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(256), 0, s, a);
  return check_launch("integrate");
}

}  // namespace kf
