// kf_device.hpp — device-side helpers shared by the gfx950 kernels.
//
// All arithmetic here is written as explicit IEEE float operations in a fixed
// order; the library is compiled with -ffp-contract=off and HIP's default
// correctly rounded fp32 division and square root, so a host restatement that
// evaluates the same expressions in the same order produces the same bits.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kinfu.h"

namespace kf {

constexpr int kWave = 64;  // CDNA wavefront width

struct f3 {
  float x, y, z;
};

__device__ __forceinline__ f3 mk(float x, float y, float z) { return f3{x, y, z}; }
__device__ __forceinline__ f3 sub(f3 a, f3 b) { return f3{a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ float dot(f3 a, f3 b) { return (a.x * b.x + a.y * b.y) + a.z * b.z; }
__device__ __forceinline__ f3 cross(f3 a, f3 b) {
  return f3{a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}

// R * v (+ t): ((r0*x + r1*y) + r2*z) + t0, row by row.
__device__ __forceinline__ f3 rot(const float* r, f3 v) {
  return f3{(r[0] * v.x + r[1] * v.y) + r[2] * v.z, (r[3] * v.x + r[4] * v.y) + r[5] * v.z,
            (r[6] * v.x + r[7] * v.y) + r[8] * v.z};
}
__device__ __forceinline__ f3 xform(const kf_posef& p, f3 v) {
  f3 a = rot(p.r, v);
  return f3{a.x + p.t[0], a.y + p.t[1], a.z + p.t[2]};
}

__device__ __forceinline__ bool finite3(f3 v) { return v.x == v.x && v.y == v.y && v.z == v.z; }

// Round half up, as x - floor(x) < 0.5 ? floor(x) : ceil(x) (result kept as float).
__device__ __forceinline__ float round_half_up(float a) {
  float fl = floorf(a);
  return (a - fl) < 0.5f ? fl : ceilf(a);
}

// e^-x for x >= 0 from a base-2 range reduction and a degree-8 Taylor
// polynomial of e^-y on y in [0, ln 2); returns 0 for x >= 80 or NaN.  Plain IEEE
// single operations only, so host and device give the same bits.
__host__ __device__ __forceinline__ float exp_neg(float x) {
  if (!(x < 80.0f)) return 0.0f;
  // n = floor(x / ln2); r = x - n ln2 by Cody-Waite (ln2_hi has 16 significant
  // bits, so n * ln2_hi and x - n * ln2_hi are exact for n < 128).
  const float n = floorf(x * 1.44269504f);
  const float y = (x - n * 0.693145752f) - n * 1.42860677e-06f;
  float p = 2.48015873e-05f;      // 1/8!
  p = p * y - 1.98412698e-04f;    // 1/7!
  p = p * y + 1.38888889e-03f;    // 1/6!
  p = p * y - 8.33333333e-03f;    // 1/5!
  p = p * y + 4.16666667e-02f;    // 1/4!
  p = p * y - 1.66666667e-01f;    // 1/3!
  p = p * y + 5.00000000e-01f;    // 1/2!
  p = p * y - 1.0f;
  p = p * y + 1.0f;
  return ldexpf(p, -(int)n);
}

__device__ __forceinline__ float nanf_() { return __builtin_nanf(""); }

// 1.0f / z for positive normal z: the hardware reciprocal and one Newton step give the IEEE
// quotient below 2^126 (tests/test_gpu_device_math.py compares every mantissa); beyond,
// where the quotient is subnormal, the division itself.
__device__ __forceinline__ float reciprocal(float z) {
  float r = __builtin_amdgcn_rcpf(z);
  r = fmaf(r, fmaf(-z, r, 1.0f), r);
  if (__builtin_expect(__any(z >= 0x1p126f), 0)) r = z >= 0x1p126f ? 1.0f / z : r;
  return r;
}

// Packed FP16 voxel: low 16 bits = half(tsdf/T), high 16 bits = uint16 weight.
__device__ __forceinline__ float half_bits_to_float(uint32_t h) {
  _Float16 v = __builtin_bit_cast(_Float16, (uint16_t)h);
  return (float)v;
}
__device__ __forceinline__ uint32_t float_to_half_bits(float f) {
  _Float16 v = (_Float16)f;  // v_cvt_f16_f32, round to nearest even
  return (uint32_t)__builtin_bit_cast(uint16_t, v);
}

// DPP lane move (GFX9 encodings): quad_perm xor1 = 0xB1, xor2 = 0x4E; row_ror:4 =
// 0x124, row_ror:8 = 0x128; row_bcast:15 = 0x142, row_bcast:31 = 0x143.  Lanes in
// rows excluded by ROW_MASK receive 0.
template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ float dpp_f(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, ROW_MASK,
                                                               0xf, false));
}
template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ int dpp_i(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, ROW_MASK, 0xf, false);
}

template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ double dpp_d(double v) {
  const long long b = __builtin_bit_cast(long long, v);
  const int lo = dpp_i<CTRL, ROW_MASK>((int)(b & 0xffffffffll));
  const int hi = dpp_i<CTRL, ROW_MASK>((int)(b >> 32));
  return __builtin_bit_cast(double, ((long long)hi << 32) | (long long)(unsigned)lo);
}

// Sum over the 64 lanes of a wavefront with DPP moves only (no LDS): quad xor
// steps, row rotations, then the two row broadcasts.  The total is in lane 63.
__device__ __forceinline__ int wave_sum_i_lane63(int v) {
  v += dpp_i<0xB1>(v);
  v += dpp_i<0x4E>(v);
  v += dpp_i<0x124>(v);
  v += dpp_i<0x128>(v);
  v += dpp_i<0x142, 0xA>(v);
  v += dpp_i<0x143, 0xC>(v);
  return v;
}

// Bitwise OR over the 64 lanes of a wavefront (DPP ladder), returned to all lanes.
__device__ __forceinline__ unsigned wave_or_u32(unsigned v) {
  int x = (int)v;
  x |= dpp_i<0xB1>(x);
  x |= dpp_i<0x4E>(x);
  x |= dpp_i<0x124>(x);
  x |= dpp_i<0x128>(x);
  x |= dpp_i<0x142, 0xA>(x);
  x |= dpp_i<0x143, 0xC>(x);
  return (unsigned)__builtin_amdgcn_readlane(x, 63);
}

// Orders the LDS accesses of one wavefront around this point.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// x returned through an empty asm statement: the compiler cannot see its range, so
// it neither widens the arithmetic that uses it to 64 bits nor fuses a 24-bit
// multiply and add into a 64-bit multiply-add.
__device__ __forceinline__ unsigned opaque_u32(unsigned x) {
  asm("" : "+v"(x));
  return x;
}

// Element at byte offset off of a plane: a uniform base address plus one 32-bit
// offset register, shared by every plane read at the same index.
__device__ __forceinline__ float plane_at(const float* p, unsigned off) {
  return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(p) + off);
}

// Brick occupancy map: `per_col` 64-bit words per brick column (bx, by), bit bz & 63
// of word (bx * nb + by) * per_col + (bz >> 6).
struct OccMap {
  unsigned long long* words;  // nb * nb * per_col
  int nb;
  int per_col;
};

// Brick occupancy (bricks of 8^3 voxels): a voxel at index z along an axis lies in
// the extended extent [8b, 8b + 8] of brick b = z >> 3 and, when z is a multiple of
// 8, of brick b - 1 as well.  Marks, in word kw of voxel column (ix, iy)'s brick
// columns, the OR of the lanes' bit sets (whole wave, uniform control flow).  Up to
// four brick columns receive the bits (the column's own and, on a brick boundary,
// the one below in x and/or y); a word is only written when bits are missing.
__device__ __forceinline__ void occ_mark_column(const OccMap& occ, int ix, int iy, int kw, unsigned long long bits,
                                                int lane) {
  if (__ballot(bits != 0ull) == 0ull) return;
  const unsigned lo = wave_or_u32((unsigned)bits);
  const unsigned hi = wave_or_u32((unsigned)(bits >> 32));
  const unsigned long long zm = ((unsigned long long)hi << 32) | lo;
  if (lane < 4) {
    const int bx0 = ix >> 3, by0 = iy >> 3;
    const int bx = (lane & 1) ? (((ix & 7) == 0 && bx0 > 0) ? bx0 - 1 : -1) : bx0;
    const int by = (lane & 2) ? (((iy & 7) == 0 && by0 > 0) ? by0 - 1 : -1) : by0;
    if (bx >= 0 && by >= 0) {
      unsigned long long* w = occ.words + ((bx * occ.nb + by) * occ.per_col + kw);
      const unsigned long long cur = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if ((cur & zm) != zm) __hip_atomic_fetch_or(w, zm, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// Wave-level sum of a float with the DPP/permute ladder, result valid in all lanes.
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, kWave);
  return v;
}
__device__ __forceinline__ int wave_sum_i(int v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, kWave);
  return v;
}

}  // namespace kf
