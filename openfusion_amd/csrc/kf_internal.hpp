// kf_internal.hpp — host-side internals of libkinfu (handle layouts, error plumbing,
// kernel launchers shared between translation units).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>

#include "kinfu.h"

namespace kf {

void set_error(const std::string& msg);
kf_status hip_fail(hipError_t e, const char* what);

#define KF_HIP(call)                                        \
  do {                                                      \
    hipError_t e_ = (call);                                 \
    if (e_ != hipSuccess) return ::kf::hip_fail(e_, #call); \
  } while (0)

#define KF_CHECK_ARG(cond, msg)                   \
  do {                                            \
    if (!(cond)) {                                \
      ::kf::set_error(std::string("invalid argument: ") + (msg)); \
      return KF_ERR_INVALID_ARGUMENT;             \
    }                                             \
  } while (0)

#define KF_TRY(call)                 \
  do {                               \
    kf_status s_ = (call);           \
    if (s_ != KF_OK) return s_;      \
  } while (0)

inline hipStream_t S(kf_stream s) { return reinterpret_cast<hipStream_t>(s); }
inline int div_up(int a, int b) { return (a + b - 1) / b; }

// Launches the last queued kernel's error check (launch-configuration errors only).
kf_status check_launch(const char* what);

}  // namespace kf

struct kf_volume {
  kf_volume_desc desc;
  void* d_voxels = nullptr;  // n^3 * voxel_bytes
  size_t bytes = 0;
  // Sweep work list, rewritten by every sweep: the counts of exact and free bricks,
  // then one word per 8^3 brick that the sweep must visit, bx << 24 | by << 16 |
  // bz << 8 | class, the exact ones from the front and the free ones from the back;
  // room for all nb^3 bricks.  And the raylen extrema of the 8x8 and 32x32 pixel
  // tiles the classes come from (sized for the largest image).
  uint32_t* d_bricks = nullptr;
  float2* d_rtiles = nullptr;
  // Brick occupancy map: bricks of 8^3 voxels, occ_words 64-bit words per (bx, by)
  // brick column, bit bz & 63 of word (bx * nb + by) * occ_words + (bz >> 6).  A
  // clear bit guarantees f == 1 for every voxel of the brick extended by one voxel
  // along +x, +y, +z (all corners of a trilinear sample whose base voxel lies in the
  // brick).  The sweep sets bits as it writes f != 1; bits are never cleared except
  // by a reset or a rebuild.
  unsigned long long* d_occ = nullptr;
  // Chebyshev distance, in bricks, from each brick to the nearest set brick bit,
  // capped at kBrickDistCap (one byte per brick, (bx * nb + by) * 64 * occ_words + bz);
  // recomputed before every raycast.
  uint8_t* d_bdist = nullptr;
  int occ_nb = 0;                // bricks per axis (0: no map)
  int occ_words = 0;             // 64-bit words per brick column: ceil(nb / 64)
  bool occ_enabled = true;       // kf_volume_set_free_space_skip: off = no map, no skip
  mutable bool occ_stale = false;  // voxels may have been written outside the library
};

// ICP scratch and per-iteration control block (device memory).
// The single-launch form's grid barrier counts arrivals in eight group counters
// (block index mod 8) and one top counter, and releases the waiting blocks through
// a generation word; the counters only grow (a call takes their values at its start
// as its base), each on a 128-byte line of its own.
struct kf_icp_ctrl {
  unsigned int poll_limit;  // single-launch barrier: polls before a wait gives up (0: the default bound)
  int executed;             // multi-launch calls: iterations that produced an update
  int broken;               // a barrier wait timed out: single-launch calls report status 2
  unsigned int pad0[29];
  unsigned int gen;         // barriers completed (advanced by the last arrival)
  unsigned int pad1[31];
  unsigned int top;         // group counters that completed a barrier
  unsigned int pad2[31];
  unsigned int group[8][32];  // arrivals of the blocks of each group (element [g][0])
};

struct kf_tracker {
  kf_intrinsics k0;
  kf_icp_params params;
  int max_blocks = 0;     // partial slots
  double* d_partials = nullptr;  // two sets of max_blocks slots of 32 doubles (terms, counts, stop marker)
  kf_icp_ctrl* d_ctrl = nullptr;
  kf_pose* d_work = nullptr;     // two poses: the step outputs alternate between them
  kf_icp_stats* d_stats_tmp = nullptr;  // used when the caller passes none
  int chain_capacity = -1;      // co-resident blocks of the single-launch kernel (-1: not queried)
  double* d_sums_tmp = nullptr;
};

namespace kf {

// Launchers implemented in the .hip translation units.  kernel_start / kernel_stop
// (optional, together): events that take the main kernel's own start and end
// times (hipExtLaunchKernelGGL).
// l2_copy (optional): a second destination of the level-2 depth, written by the same
// kernel (the frame driver's learned-prior input slot).
kf_status launch_preprocess(const kf_intrinsics& k0, const kf_preprocess_params& p,
                            const uint16_t* d_depth, kf_frame_maps& live, hipStream_t s, float* l2_copy = nullptr);
kf_status launch_volume_reset(kf_volume* v, hipStream_t s);
// Raylen tiles of a depth frame made ahead of its sweep (the frame driver makes them
// on its side stream while the previous frame's sweep runs): the 8x8 tiles, then
// the 32x32 ones (sweep_tiles_floats2 float2 for the image), and the two counts
// (exact, free) of the sweep's work list, which launch_raylen_tiles zeroes.
struct SweepTiles {
  float2* tiles;
  uint32_t* count;
};
size_t sweep_tiles_floats2(const kf_intrinsics& k0);
kf_status launch_raylen_tiles(const kf_intrinsics& k0, const float* d_raylen, const SweepTiles& t, hipStream_t s);
// pre: the tiles of d_raylen from launch_raylen_tiles (nullptr: made here).
kf_status launch_integrate(kf_volume* v, const kf_intrinsics& k0, const kf_integrate_params& p,
                           const float* d_raylen, const kf_pose* d_pose,
                           unsigned long long* d_updated, uint32_t* d_mask, hipStream_t s,
                           hipEvent_t between = nullptr, hipEvent_t kernel_start = nullptr,
                           hipEvent_t kernel_stop = nullptr, const SweepTiles* pre = nullptr);
kf_status launch_volume_stats(const kf_volume* v, double* d_out, hipStream_t s);
// Recomputes the occupancy map from the voxels when it is stale (no-op otherwise).
kf_status ensure_occupancy(const kf_volume* v, hipStream_t s);
// Brick distances from the current occupancy map (no-op without a map).
constexpr int kBrickDistCap = 16;
kf_status launch_brick_distance(const kf_volume* v, hipStream_t s);
constexpr int kOccWordBricks = 64;  // bricks held in one 64-bit occupancy word
// Words per brick column of a volume with n voxels per axis (n <= 2048: at most 4).
inline int occ_words_for(int n) { return (n / 8 + kOccWordBricks - 1) / kOccWordBricks; }
constexpr int kMaxImage = 8192;    // largest image side accepted by the API
// raylen tiles: 8x8 then 32x32 pixels, (min, max) per tile
constexpr size_t kRayTiles8 = (size_t)(kMaxImage / 8) * (kMaxImage / 8);
constexpr size_t kRayTiles = kRayTiles8 + (size_t)(kMaxImage / 32) * (kMaxImage / 32);
kf_status launch_raycast(const kf_volume* v, const kf_intrinsics& k0, const kf_raycast_params& p,
                         const kf_pose* d_pose, kf_frame_maps& model, unsigned long long* d_steps,
                         hipStream_t s, hipEvent_t after_distances = nullptr,
                         unsigned long long* d_diag = nullptr, hipEvent_t kernel_start = nullptr,
                         hipEvent_t kernel_stop = nullptr);
// Acceptance test of a warm-started tracking call, evaluated at the end of that
// call: it fails when the call reports an error, ran no iteration or has a NaN
// residual, when fewer than min_frac of the candidates are inliers, or (once
// window_min residuals are known) when its residual exceeds ratio x the median of
// the window.  Passed: *accept_out <- the call's pose and fallback->skip = 1;
// failed: fallback->skip = 0.  *used <- 1, *fell_back <- failed.
constexpr int kGateMaxWindow = 64;
struct IcpGate {
  const double* window;    // recent accepted residuals (window_len entries)
  const int32_t* count;    // how many of them are valid
  int window_len;          // <= kGateMaxWindow
  kf_icp_stats* fallback;  // skip flag of the fallback call
  kf_pose* accept_out;
  int32_t* used;
  int32_t* fell_back;
  float ratio, min_frac;
  int window_min;
};
struct FrameEnd;  // kf_frame_end.hpp
// single_launch: the whole call as one launch (also when the tracker's parameters
// do not ask for it); used where most calls are skipped by the statistics' flag.
// gate (multi-launch calls only): evaluated by the call's last kernel.
// frame_end: the frame driver's end-of-frame bookkeeping, run by the call's last
// kernel once the pose is final (also when the call is skipped).
kf_status launch_icp_track(kf_tracker* t, const kf_frame_maps& live, const kf_frame_maps& model,
                           const kf_pose* d_guess, kf_pose* d_out, kf_icp_stats* d_stats,
                           hipStream_t s, bool single_launch = false, const IcpGate* gate = nullptr,
                           const FrameEnd* frame_end = nullptr);
// kf_icp_track_noalloc: launch_icp_track over the library's static scratch.
kf_status launch_icp_track_noalloc(const kf_intrinsics& k0, const kf_icp_params& p, const kf_frame_maps& live,
                                   const kf_frame_maps& model, const kf_pose* d_guess, kf_pose* d_out,
                                   kf_icp_stats* d_stats, hipStream_t s);
kf_status launch_icp_reduce(kf_tracker* t, int level, const kf_frame_maps& live,
                            const kf_frame_maps& model, const kf_pose* d_est, double* d_sums,
                            uint8_t* d_mask, hipStream_t s);
kf_status launch_pose_constant_velocity(const kf_pose* d_prev2, const kf_pose* d_prev1,
                                        kf_pose* d_guess, hipStream_t s);
kf_status launch_pose_copy(const kf_pose* d_src, kf_pose* d_dst, hipStream_t s);

// Host-side FP64 pose helpers (identical operation order to the device versions).
void pose_finish(kf_pose* p);  // fills wc / cw from T_wc

}  // namespace kf
