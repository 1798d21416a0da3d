// kf_prior_net.hpp — the learned pose prior's network: shapes, parameter layout and the
// device helpers that its inference and training kernels share.
#pragma once

#include "kf_device.hpp"
#include "kf_internal.hpp"

namespace kf {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

// One 16x16x32 BF16 MFMA step (gfx950): lane l supplies A(l % 16, k0 + 8 (l / 16) + j)
// and B(k0 + 8 (l / 16) + j, l % 16) for j < 8 as one 16-byte vector each, and holds
// C(4 (l / 16) + j, l % 16) for j < 4.
__device__ __forceinline__ v4f mfma32(uint4 a, uint4 b, v4f acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), acc, 0,
                                                 0, 0);
}

constexpr int kH0 = KF_PRIOR_HEIGHT, kW0 = KF_PRIOR_WIDTH;
constexpr int kConvs = 4;
constexpr int kFeat = 128, kTwist = 6, kFc1In = kFeat + kTwist, kHidden = 256;

struct ConvShape {
  int cin, cout, hin, win, hout, wout, kc;
};
constexpr ConvShape kConv[kConvs] = {
    {2, 32, 120, 160, 60, 80, 18},
    {32, 64, 60, 80, 30, 40, 288},
    {64, 64, 30, 40, 15, 20, 576},
    {64, 128, 15, 20, 8, 10, 576},
};
constexpr int kPool = 8 * 10;

// Parameter blob offsets (floats).
struct ParamLayout {
  long w[6], b[6], total;
  ParamLayout() {
    long o = 0;
    for (int l = 0; l < kConvs; ++l) {
      w[l] = o;
      o += (long)kConv[l].cout * kConv[l].kc;
      b[l] = o;
      o += kConv[l].cout;
    }
    w[4] = o;
    o += (long)kHidden * kFc1In;
    b[4] = o;
    o += kHidden;
    w[5] = o;
    o += (long)kTwist * kHidden;
    b[5] = o;
    o += kTwist;
    total = o;
  }
};
inline const ParamLayout& layout() {
  static const ParamLayout L;
  return L;
}

// Position of element (row, k) in an operand copy of a weight matrix of `rows` rows: a
// lane's operand vector is eight k of one row, and the lanes of a quarter wave read
// neighbouring rows of the same k, so the rows of a vector position lie together.  (Rows on
// end: a quarter wave's sixteen vectors lie on sixteen lines, and the L1 looks each up:
// inference at batch 1 17.6 us instead of 12.0, gradients at batch 19 84 instead of 69.)
__host__ __device__ __forceinline__ int operand_at(int rows, int row, int k) { return ((k >> 3) * rows + row) * 8 + (k & 7); }

// Rounds to the nearest BF16, ties to even: v_cvt_pk_bf16_f32, one instruction for two
// values (as integer arithmetic on their bits, about nine; the bits are the same for every
// number and the usual quiet NaN).
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f{lo, hi}), v2bf));
}
__device__ __forceinline__ uint16_t bf16_rne(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

}  // namespace kf
