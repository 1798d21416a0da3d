// kf_preprocess.hip — depth conditioning for one frame on gfx950.
//
// Replaces d_convertDepthToWorldVertices / d_convertDepthToWorldNormals
// (Source/src/CameraSupport/CameraHandler.cu:65-132) and adds the bilateral
// filter and 3-level pyramid the reference only mentions (CameraHandler.cu:6).
// Maps are kept in the camera frame; the tracker applies the pose itself.
//
//   depth_levels  : uint16 -> metres, range gate, raylen = |K^-1 [x,y,1]| * d,
//                   bilateral filter (LDS tile with halo, spatial weights
//                   from the kernel arguments, range weights from a
//                   per-block LDS table); then levels 1 and 2 from the block's
//                   filtered tile in LDS: 2x2 block average gated by
//                   |d - centre| < gate                       [two L0 pixels]
//   vertex_normal : v = d * K^-1 [x,y,1];  n = normalize((v(x,y+1)-v) x (v(x+1,y)-v))
//                   (points towards the camera), all levels in one launch
#include <type_traits>

#include "kf_device.hpp"
#include "kf_internal.hpp"

namespace kf {
namespace {

constexpr int kTileX = 32, kTileY = 16;  // level-0 pixels of a block
constexpr int kThreads = kTileX * kTileY / 2;
constexpr int kMaxRadius = 4;

struct PreArgs {
  const uint16_t* depth;
  float* raylen;
  float* out;  // filtered level-0 depth
  float *l1, *l2, *l2_copy;  // filtered depth of levels 1 and 2 (NULL: no such level) and a copy of level 2
  int W1, H1, W2, H2;
  float gate;
  int W, H;
  float fx, fy, cx, cy;
  float scale, dmin, dmax;
  float inv2sr;  // 0.5/sigma_r^2
  // spatial weight of each window offset, row-major (2 radius + 1)^2, made on the
  // host with the same exp_neg (kernel arguments: scalar registers in the kernel)
  float ws[(2 * kMaxRadius + 1) * (2 * kMaxRadius + 1)];
};

// One coarse pixel: the mean of the valid samples of its 2x2 block (those inside
// the fine level) within `gate` of the block's top-left sample, 0 when that one is
// invalid.  get(sx, sy): the fine sample.
template <typename Get>
__device__ __forceinline__ float pyr_pixel(const Get& get, int x, int y, int Wi, int Hi, float gate) {
  const float c = get(2 * x, 2 * y);
  float r = 0.0f;
  if (c != 0.0f) {
    float s = 0.0f, n = 0.0f;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int sx = 2 * x + i, sy = 2 * y + j;
        if (sx >= Wi || sy >= Hi) continue;
        const float d = get(sx, sy);
        if (d > 0.0f && fabsf(d - c) < gate) {
          s = s + d;
          n = n + 1.0f;
        }
      }
    }
    r = s / n;
  }
  return r;
}

// Bilateral weight of a neighbour: exp(-|dp|^2 / 2 sigma_s^2) * exp(-dr^2 / 2 sigma_r^2)
// with dr = |u_q - u_c| * scale (the integer depth-code difference in metres).  Both
// factors are exp_neg values: the spatial ones made on the host (kernel arguments),
// the range ones in a per-block LDS table for code differences below kRangeLut.
// ZT: the range weight is exactly 0 from kRangeLut on (exp_neg's argument,
// monotone in the difference, has reached 80 there), so larger differences need no
// exp_neg of their own: the table ends with a 0 that they all read.
constexpr int kRangeLut = 512;
// Codes are held times four, so that a difference is the table's byte offset; an invalid
// pixel's is farther than any table entry from every valid one.
constexpr int kInvalid = 1 << 24;

// |a - b| in one instruction.
__device__ __forceinline__ unsigned abs_diff(unsigned a, unsigned b) {
  unsigned d;
  asm("v_sad_u32 %0, %1, %2, 0" : "=v"(d) : "v"(a), "v"(b));
  return d;
}

// A block filters kTileX x kTileY pixels, a pair of neighbours per thread (the 2R + 2
// codes of a window row are read once for both), and makes the coarser levels' pixels
// under them (tiles start at multiples of 4, so they need no other block's).  R: the
// window half-size, fixed per instance so that a window row's loop unrolls.
// Pixels outside the image are invalid in the tile, so the window needs no bounds test
// of its own; an invalid tap has weight 0, which adds exactly nothing (sums are >= 0).
//
// Bound by latency: waiting (the frame's first touch, the LDS reads, the barriers before the
// coarser levels) is half of a wavefront's life.  In one launch and with a window row's codes
// and metres read once for two pixels; kf_preprocess with three levels, against a pixel per
// thread and a second launch for the coarser levels: radius 3 640x480 13.9 / 18.5 us, 319x241
// 10.2 / 16.1, 1280x960 37.2 / 40.8.  A table of weight products per window distance (no
// products per tap) took as long.
//
// kUnroll: the window's rows unrolled, the compiler loads all of them first, which takes
// registers (radius 3: 167, three waves per SIMD); as a loop every instance has eight waves.
// Where the range weights do not end in the table, or at radius 4, the loop is far ahead:
// radius 4 640x480 15.2 us (unrolled 20.0, before 22.1), 2560x1440 77 (133, 126); weights
// beyond the table, 640x480 radius 4 19.7 (40, 23.8), 1280x960 radius 3 34.5 (47, 42.6).  At
// the frame driver's radius 3 it is too when alone (640x480 13.4 us), but beside the raycast
// its many waves take the CU slots that the raycast waits for: 512^3 stream 4,466 frames/s
// against 4,560.
template <int R, bool ZT>
__global__ __launch_bounds__(kThreads) void depth_levels(PreArgs a) {
  constexpr int kUnroll = ZT && R <= 3 ? 2 * R + 1 : 1;
  constexpr int kSpanX = kTileX + 2 * R, kSpanY = kTileY + 2 * R, kSpan = kSpanX * kSpanY;
  __shared__ __align__(8) int tile[kSpan];      // four times the depth codes
  __shared__ __align__(8) float metres[kSpan];  // the same in metres, 0 = invalid
  __shared__ float wr[kRangeLut + 1], s_xn[kTileX], s_yn[kTileY];
  __shared__ float t0[kTileY][kTileX], t1[kTileY / 2][kTileX / 2];
  const int bx = blockIdx.x * kTileX, by = blockIdx.y * kTileY;
  const int tid = threadIdx.x;
  // the tile and its halo, a row per wavefront and pass, every load of a thread in flight
  // at once (out-of-image entries read a clamped pixel and are dropped)
  constexpr int kWaves = kThreads / kWave, kPer = (kSpanY + kWaves - 1) / kWaves;
  static_assert(kSpanX <= kWave, "a row per wavefront");
  const int lane = tid & (kWave - 1), wave = tid / kWave;
  const int gx = bx + lane - R;
  const bool col = gx >= 0 && gx < a.W;
  int uv[kPer];
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int gy = by + wave + j * kWaves - R;
    const int u = a.depth[min(max(gy, 0), a.H - 1) * a.W + min(max(gx, 0), a.W - 1)];
    uv[j] = col && gy >= 0 && gy < a.H ? u : 0;
  }
  for (int i = tid; i <= kRangeLut; i += kThreads) {
    const float rm = (float)i * a.scale;
    wr[i] = i < kRangeLut ? exp_neg((rm * rm) * a.inv2sr) : 0.0f;
  }
  if (tid < kTileX)
    s_xn[tid] = ((float)(bx + tid) - a.cx) / a.fx;
  else if (tid < kTileX + kTileY)
    s_yn[tid - kTileX] = ((float)(by + tid - kTileX) - a.cy) / a.fy;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int ty = wave + j * kWaves;
    if (lane < kSpanX && ty < kSpanY) {
      const float d = (float)uv[j] * a.scale;
      const bool ok = uv[j] != 0 && d >= a.dmin && d <= a.dmax;
      tile[ty * kSpanX + lane] = ok ? 4 * uv[j] : kInvalid;
      metres[ty * kSpanX + lane] = ok ? d : 0.0f;
    }
  }
  __syncthreads();
  const int px = 2 * (tid % (kTileX / 2)), py = tid / (kTileX / 2);  // the pair's first pixel in the tile
  int uc[2];
  float sw[2] = {0.0f, 0.0f}, swd[2] = {0.0f, 0.0f};
#pragma unroll
  for (int p = 0; p < 2; ++p) uc[p] = tile[(py + R) * kSpanX + px + p + R];
#pragma unroll kUnroll
  for (int dy = -R; dy <= R; ++dy) {
    int u[2 * R + 2];
    float m[2 * R + 2];
    const int row = (py + R + dy) * kSpanX + px;
#pragma unroll
    for (int i = 0; i < 2 * R + 2; i += 2) {
      const int2 u2 = *reinterpret_cast<const int2*>(&tile[row + i]);
      const float2 m2 = *reinterpret_cast<const float2*>(&metres[row + i]);
      u[i] = u2.x;
      u[i + 1] = u2.y;
      m[i] = m2.x;
      m[i + 1] = m2.y;
    }
#pragma unroll
    for (int dx = -R; dx <= R; ++dx) {
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int uq = u[dx + R + p];
        const unsigned du4 = abs_diff((unsigned)uq, (unsigned)uc[p]);
        float w_r = *reinterpret_cast<const float*>(reinterpret_cast<const char*>(wr) + min(du4, 4u * kRangeLut));
        if (!ZT && du4 >= 4u * kRangeLut && uq != kInvalid) {
          const float rm = (float)(du4 / 4u) * a.scale;
          w_r = exp_neg((rm * rm) * a.inv2sr);
        }
        const float w = a.ws[(dy + R) * (2 * R + 1) + (dx + R)] * w_r;
        sw[p] = sw[p] + w;
        swd[p] = swd[p] + w * m[dx + R + p];
      }
    }
  }
  const int x = bx + px, y = by + py;
  const float yn = s_yn[py];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const bool ok = uc[p] != kInvalid;
    const float f = ok ? swd[p] / sw[p] : 0.0f;
    t0[py][px + p] = f;
    if (x + p < a.W && y < a.H) {
      const float xn = s_xn[px + p];
      const float lam = sqrtf((xn * xn + yn * yn) + 1.0f);
      const int idx = y * a.W + x + p;
      a.raylen[idx] = ok ? metres[(py + R) * kSpanX + px + p + R] * lam : 0.0f;
      a.out[idx] = f;
    }
  }
  if (!a.l1) return;  // uniform
  __syncthreads();
  if (tid < kThreads / 2) {
    const int tx = tid % (kTileX / 2), ty = tid / (kTileX / 2);
    const int x1 = bx / 2 + tx, y1 = by / 2 + ty;
    float r = 0.0f;
    if (x1 < a.W1 && y1 < a.H1) {
      r = pyr_pixel([&](int sx, int sy) { return t0[sy - by][sx - bx]; }, x1, y1, a.W, a.H, a.gate);
      a.l1[y1 * a.W1 + x1] = r;
    }
    t1[ty][tx] = r;
  }
  if (!a.l2) return;  // uniform
  __syncthreads();
  if (tid < kThreads / 8) {
    const int tx = tid % (kTileX / 4), ty = tid / (kTileX / 4);
    const int x2 = bx / 4 + tx, y2 = by / 4 + ty;
    if (x2 < a.W2 && y2 < a.H2) {
      const float r = pyr_pixel([&](int sx, int sy) { return t1[sy - by / 2][sx - bx / 2]; }, x2, y2, a.W1, a.H1, a.gate);
      a.l2[y2 * a.W2 + x2] = r;
      if (a.l2_copy) a.l2_copy[y2 * a.W2 + x2] = r;
    }
  }
}

constexpr int kMapX = 64, kMapY = 4;

struct LevelMapArgs {
  const float* depth;
  float *vx, *vy, *vz, *nx, *ny, *nz;
  int W, H;
  float fx, fy, cx, cy;
  int block_begin;  // first linear block of this level
  int blocks_x;
};
struct MapArgs {
  LevelMapArgs lv[KF_MAX_LEVELS];
  int levels;
};

// Vertices and normals, one pixel per thread, a wavefront per kMapX pixels of a row (its
// six planes' stores are whole lines).  x and y in camera units are divided once per
// block, not four times per pixel.  Bound by its stores; 640x480 and two coarser levels:
// 4.8 us (16x16 blocks that divided per pixel: 6.1).
__global__ __launch_bounds__(kMapX * kMapY) void vertex_normal(MapArgs m) {
  __shared__ float s_xn[kMapX + 1], s_yn[kMapY + 1];
  int b = blockIdx.x;
  int l = 0;
  for (int i = 1; i < m.levels; ++i)
    if (b >= m.lv[i].block_begin) l = i;
  const LevelMapArgs& a = m.lv[l];
  b -= a.block_begin;
  const int by = b / a.blocks_x, bx = b - by * a.blocks_x;
  const int tx = threadIdx.x % kMapX, ty = threadIdx.x / kMapX;
  const int x = bx * kMapX + tx, y = by * kMapY + ty;
  // the pixel's depth and its right and lower neighbours' (clamped, dropped at the edges)
  const bool in = x < a.W && y < a.H, edge = x + 1 >= a.W || y + 1 >= a.H;
  const int idx = in ? y * a.W + x : 0;
  const float d = a.depth[idx], dr = a.depth[edge ? idx : idx + 1], dd = a.depth[edge ? idx : idx + a.W];
  for (int i = threadIdx.x; i < kMapX + kMapY + 2; i += kMapX * kMapY) {
    if (i <= kMapX)
      s_xn[i] = ((float)(bx * kMapX + i) - a.cx) / a.fx;
    else
      s_yn[i - kMapX - 1] = ((float)(by * kMapY + i - kMapX - 1) - a.cy) / a.fy;
  }
  __syncthreads();
  if (!in) return;
  const float xn = s_xn[tx], yn = s_yn[ty];
  f3 v = f3{nanf_(), nanf_(), nanf_()}, n = v;
  if (d != 0.0f) {
    v = f3{xn * d, yn * d, d};
    if (!edge && dr != 0.0f && dd != 0.0f) {
      const f3 vr = f3{s_xn[tx + 1] * dr, yn * dr, dr}, vd = f3{xn * dd, s_yn[ty + 1] * dd, dd};
      const f3 c = cross(sub(vd, v), sub(vr, v));
      const float len = sqrtf(dot(c, c));
      if (len > 0.0f) {
        const float inv = 1.0f / len;
        n = f3{c.x * inv, c.y * inv, c.z * inv};
      }
    }
  }
  a.vx[idx] = v.x;
  a.vy[idx] = v.y;
  a.vz[idx] = v.z;
  a.nx[idx] = n.x;
  a.ny[idx] = n.y;
  a.nz[idx] = n.z;
}

}  // namespace

kf_status launch_preprocess(const kf_intrinsics& k0, const kf_preprocess_params& p,
                            const uint16_t* d_depth, kf_frame_maps& live, hipStream_t s, float* l2_copy) {
  KF_CHECK_ARG(d_depth != nullptr, "depth is NULL");
  KF_CHECK_ARG(!l2_copy || live.levels > 2, "a level-2 copy needs three levels");
  KF_CHECK_ARG(live.levels >= 1 && live.levels <= KF_MAX_LEVELS, "levels must be 1..3");
  KF_CHECK_ARG(p.bilateral_radius >= 0 && p.bilateral_radius <= kMaxRadius, "bilateral_radius must be 0..4");
  KF_CHECK_ARG(p.sigma_space_px > 0.0f && p.sigma_range_m > 0.0f, "sigmas must be positive");
  KF_CHECK_ARG(live.raylen != nullptr, "live.raylen is NULL");
  for (int l = 0; l < live.levels; ++l) {
    const kf_level_maps& m = live.level[l];
    kf_intrinsics kl = kf_intrinsics_level(&k0, l);
    KF_CHECK_ARG(m.width == kl.width && m.height == kl.height, "map level size mismatch");
    KF_CHECK_ARG(m.depth && m.vx && m.vy && m.vz && m.nx && m.ny && m.nz, "map plane is NULL");
  }
  PreArgs a;
  a.depth = d_depth;
  a.raylen = live.raylen;
  a.out = live.level[0].depth;
  a.W = k0.width;
  a.H = k0.height;
  a.fx = k0.fx;
  a.fy = k0.fy;
  a.cx = k0.cx;
  a.cy = k0.cy;
  a.scale = p.depth_scale;
  a.dmin = p.min_depth_m;
  a.dmax = p.max_depth_m;
  const float inv2ss = 0.5f / (p.sigma_space_px * p.sigma_space_px);
  a.inv2sr = 0.5f / (p.sigma_range_m * p.sigma_range_m);
  const int R = p.bilateral_radius;
  for (int dy = -R; dy <= R; ++dy)
    for (int dx = -R; dx <= R; ++dx)
      a.ws[(dy + R) * (2 * R + 1) + (dx + R)] = exp_neg((float)(dx * dx + dy * dy) * inv2ss);
  const float rm_lut = (float)kRangeLut * a.scale;
  const bool zt = exp_neg((rm_lut * rm_lut) * a.inv2sr) == 0.0f;
  const bool one = live.levels > 1, two = live.levels > 2;
  a.l1 = one ? live.level[1].depth : nullptr;
  a.l2 = two ? live.level[2].depth : nullptr;
  a.l2_copy = two ? l2_copy : nullptr;
  a.W1 = one ? live.level[1].width : 0;
  a.H1 = one ? live.level[1].height : 0;
  a.W2 = two ? live.level[2].width : 0;
  a.H2 = two ? live.level[2].height : 0;
  a.gate = p.pyramid_gate_m;
  const dim3 grd(div_up(k0.width, kTileX), div_up(k0.height, kTileY));
  auto pick = [&](auto zt_tag) {
    constexpr bool Z = decltype(zt_tag)::value;
    switch (R) {
      case 0: return depth_levels<0, Z>;
      case 1: return depth_levels<1, Z>;
      case 2: return depth_levels<2, Z>;
      case 3: return depth_levels<3, Z>;
      default: return depth_levels<4, Z>;
    }
  };
  auto kern = zt ? pick(std::true_type{}) : pick(std::false_type{});
  hipLaunchKernelGGL(kern, grd, dim3(kThreads), 0, s, a);
  KF_TRY(check_launch("depth_levels"));

  MapArgs m;
  int blocks = 0;
  m.levels = live.levels;
  for (int l = 0; l < live.levels; ++l) {
    kf_intrinsics kl = kf_intrinsics_level(&k0, l);
    LevelMapArgs& la = m.lv[l];
    const kf_level_maps& lm = live.level[l];
    la.depth = lm.depth;
    la.vx = lm.vx; la.vy = lm.vy; la.vz = lm.vz;
    la.nx = lm.nx; la.ny = lm.ny; la.nz = lm.nz;
    la.W = kl.width; la.H = kl.height;
    la.fx = kl.fx; la.fy = kl.fy; la.cx = kl.cx; la.cy = kl.cy;
    la.blocks_x = div_up(kl.width, kMapX);
    la.block_begin = blocks;
    blocks += la.blocks_x * div_up(kl.height, kMapY);
  }
  hipLaunchKernelGGL(vertex_normal, dim3(blocks), dim3(kMapX * kMapY), 0, s, m);
  return check_launch("vertex_normal");
}

}  // namespace kf
