/*
 * kinfu.h — C ABI of the MI355X (gfx950) KinectFusion hot path.
 *
 * Every entry point is `extern "C"`, takes plain pointers and sizes, returns a
 * kf_status (never exits the process) and is asynchronous on the stream it is
 * given (NULL = the device's default stream) unless its comment says "blocking".
 * Handles are thread-compatible (one handle per host thread), not thread-safe.
 *
 * Units: metres, seconds, pixels.  Camera frame: x right, y down, z forward
 * (standard pinhole).  Poses are row-major 4x4, T_wc maps camera -> world.
 *
 * Each group names the reference interface it replaces (paths relative to the
 * OpenFusion source tree).
 */
#ifndef KINFU_H_
#define KINFU_H_

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* ------------------------------------------------------------------------ */
/* Status codes.  Replace cutilSafeCall's print-and-exit
 * (Source/include/Utils/cutil_inline_runtime.h:256-263). */
typedef enum kf_status {
  KF_OK = 0,
  KF_ERR_INVALID_ARGUMENT = 1,
  KF_ERR_HIP = 2,
  KF_ERR_OUT_OF_MEMORY = 3,
  KF_ERR_NOT_READY = 4,
  KF_ERR_IO = 5,
  KF_ERR_UNSUPPORTED = 6
} kf_status;

typedef void* kf_stream; /* a hipStream_t; NULL = default stream */

/* Last error text of the calling thread (never NULL). */
const char* kf_last_error(void);

/* ------------------------------------------------------------------------ */
/* Core types.  Replace CameraParams / Intrinsic (Source/include/BasicTypes.h:74-103)
 * and the compile-time constants of Source/include/Constants.h:10-55. */
typedef struct kf_intrinsics {
  float fx, fy, cx, cy; /* pixels; pixel (x,y) centre is at integer coordinates */
  int32_t width, height;
} kf_intrinsics;

/* Intrinsics of pyramid level `level` (2^level downsampling, pixel-centre aligned). */
kf_intrinsics kf_intrinsics_level(const kf_intrinsics* k0, int32_t level);

typedef enum kf_voxel_format {
  KF_VOXEL_F32 = 0, /* 8 B/voxel: {float tsdf/T, float weight}            */
  KF_VOXEL_F16 = 1  /* 4 B/voxel: {half tsdf/T (low 16 bits), u16 weight} */
} kf_voxel_format;

/* Volume: n^3 voxels, z fastest (index = (x*n + y)*n + z), voxel (i,j,k) centre at
 * origin + (i+0.5, j+0.5, k+0.5) * extent/n.  Replaces the tsdf/weight pair
 * allocated in RunApp::initCudaPointers (Source/src/MainApp.cpp:596-597). */
typedef struct kf_volume_desc {
  int32_t n;
  float extent_m;
  float origin_m[3];
  float trunc_m;
  float max_weight;
  int32_t format; /* kf_voxel_format */
} kf_volume_desc;

typedef struct kf_volume kf_volume;

/* Device pose.  Replaces d_currentTransform / d_invCurrentTransform /
 * d_cameraPosition (Source/src/MainApp.cpp:613-633).  Lives in device memory;
 * T_wc is authoritative (FP64), wc/cw are its FP32 roundings used by kernels. */
typedef struct kf_posef {
  float r[9]; /* row-major rotation */
  float t[3];
} kf_posef;

typedef struct kf_pose {
  double T_wc[16]; /* camera -> world, row-major, FP64 */
  kf_posef wc;     /* (float) of T_wc's upper 3x4                          */
  kf_posef cw;     /* (float) of the FP64 rigid inverse (R^T, -R^T t)        */
} kf_pose;

/* One pyramid level of a depth / vertex / normal map set (planar SoA, row-major,
 * width*height floats each).  Invalid vertex/normal = NaN in every component;
 * invalid depth = 0.  Replaces CameraData / PointInfo (Source/include/BasicTypes.h:43-52). */
typedef struct kf_level_maps {
  int32_t width, height;
  float* depth; /* metres (live maps only; NULL in model maps) */
  float *vx, *vy, *vz;
  float *nx, *ny, *nz;
} kf_level_maps;

#define KF_MAX_LEVELS 3

typedef struct kf_frame_maps {
  int32_t levels;
  float* raylen; /* level 0 only: distance camera->measured surface along the pixel ray, 0 = invalid */
  kf_level_maps level[KF_MAX_LEVELS];
} kf_frame_maps;

/* ------------------------------------------------------------------------ */
/* Device memory and streams (for callers without their own HIP runtime binding). */
kf_status kf_device_count(int32_t* count);
kf_status kf_device_malloc(void** d_ptr, size_t bytes);
kf_status kf_device_free(void* d_ptr);
kf_status kf_host_malloc_pinned(void** h_ptr, size_t bytes);
kf_status kf_host_free_pinned(void* h_ptr);
kf_status kf_memcpy_htod(void* d_dst, const void* h_src, size_t bytes, kf_stream s);
kf_status kf_memcpy_dtoh(void* h_dst, const void* d_src, size_t bytes, kf_stream s);
kf_status kf_memcpy_dtod(void* d_dst, const void* d_src, size_t bytes, kf_stream s);
kf_status kf_memset_d8(void* d_dst, int value, size_t bytes, kf_stream s);
kf_status kf_stream_create(kf_stream* out);
kf_status kf_stream_destroy(kf_stream s);
kf_status kf_stream_synchronize(kf_stream s); /* blocking */
kf_status kf_device_synchronize(void);        /* blocking */

/* Timing events (hipEvent) recorded on the stream the kernels run on. */
typedef void* kf_event;
kf_status kf_event_create(kf_event* out);
kf_status kf_event_destroy(kf_event e);
kf_status kf_event_record(kf_event e, kf_stream s);
kf_status kf_event_elapsed_ms(kf_event start, kf_event stop, float* ms); /* blocking */

/* ------------------------------------------------------------------------ */
/* Maps: caller-owned structs of device pointers (allocated here for convenience). */
kf_status kf_maps_alloc(const kf_intrinsics* k0, int32_t levels, int32_t with_depth, kf_frame_maps* out);
kf_status kf_maps_free(kf_frame_maps* maps);

/* ------------------------------------------------------------------------ */
/* Poses.  Replaces General::UpdateTransforms' host Eigen inverse + d_updateTransforms
 * (Source/src/General.cpp:14-40, Source/src/General.cu:57-62). */
kf_status kf_pose_upload(kf_pose* d_pose, const double T_wc[16], kf_stream s);
kf_status kf_pose_download(double T_wc[16], const kf_pose* d_pose, kf_stream s); /* blocking */
/* Host helper: fills the FP32 fields of a host kf_pose from its T_wc. */
void kf_pose_finish_host(kf_pose* h_pose);

/* ------------------------------------------------------------------------ */
/* Volume.  kf_volume_reset replaces General::InitVoxelArray / d_initVoxelArray
 * (Source/src/General.cpp:42-49, Source/src/General.cu:27-50): tsdf = +1 (i.e. +T), w = 0. */
kf_status kf_volume_create(const kf_volume_desc* desc, kf_volume** out);
kf_status kf_volume_destroy(kf_volume* vol);
kf_status kf_volume_reset(kf_volume* vol, kf_stream s);
kf_status kf_volume_get_desc(const kf_volume* vol, kf_volume_desc* desc);
/* Raw voxels (layout: voxel (x,y,z) at (x*n + y)*n + z, 8-byte {f32 f, f32 w} or
 * 4-byte {f16 f, u16 w}, f = tsdf / T).  Handing out the pointer marks the brick
 * occupancy map stale (the next raycast rebuilds it); a caller that keeps the pointer
 * and writes through it later calls kf_volume_mark_modified before raycasting. */
kf_status kf_volume_data(const kf_volume* vol, void** d_voxels, size_t* bytes);
/* Read-only view of the same voxels (leaves the occupancy map as it is). */
kf_status kf_volume_data_const(const kf_volume* vol, const void** d_voxels, size_t* bytes);
kf_status kf_volume_mark_modified(kf_volume* vol);
/* Brick occupancy map used by the raycaster to skip free space (bricks of 8^3
 * voxels, nb = bricks_per_axis = n / 8, W = ceil(nb / 64) 64-bit words per brick
 * column): bit bz % 64 of word (bx*nb + by)*W + bz / 64 clear => every voxel
 * (x,y,z) with x in [8bx, 8bx+8], y in [8by, 8by+8], z in [8bz, 8bz+8] has f == 1.
 * No counterpart in the reference (its raycaster marches every step).  Rebuilds a
 * stale map on stream s first.  NULL / 0 while the free-space skip is off. */
kf_status kf_volume_occupancy(const kf_volume* vol, const uint64_t** d_words, int32_t* bricks_per_axis,
                              kf_stream s);
/* Brick distances behind the raycaster's free-space skip:
 * d_dist[(bx*nb + by)*64*W + bz] = min(Chebyshev distance in bricks to the nearest
 * set brick of the occupancy map, 16), computed from the current map (enqueued on
 * s).  No counterpart in the reference (it marches every step); NULL / 0 while the
 * free-space skip is off. */
kf_status kf_volume_brick_distance(const kf_volume* vol, const uint8_t** d_dist, int32_t* bricks_per_axis,
                                   kf_stream s);
/* Switches the occupancy map and the raycaster's free-space skip on (1, the
 * default) or off (0: the sweep maintains no map and the raycaster samples every
 * step).  Raycast results are the same either way; off is for tests and timing.
 * Switched back on, the map is rebuilt from the voxels before its next use. */
kf_status kf_volume_set_free_space_skip(kf_volume* vol, int32_t on);
/* Occupancy statistics over every voxel (reads the whole volume once):
 * d_out (device, 4 doubles) = {observed voxels (w > 0), sum of w, sum of f over
 * observed voxels, voxels with f < 0 and w > 0}. */
kf_status kf_volume_stats(const kf_volume* vol, double* d_out, kf_stream s);

/* Raw tsdf export (replaces RunApp::saveVolumeToFile, Source/src/MainApp.cpp:181-275):
 * d_out (device, n^3 floats) = tsdf in metres in the reference's x*n^2 + y*n + z
 * order; unobserved voxels read +T. */
kf_status kf_volume_export_tsdf(const kf_volume* vol, float* d_out, kf_stream s);
/* Surface extraction by marching tetrahedra (the reference has only a disabled
 * marching-cubes sketch, Source/src/MainApp.cpp:277-328).  Writes up to max_tris
 * triangles (9 floats each: three world-space vertices, facing free space) to
 * d_tris and the number found (may exceed max_tris) to *d_count (device uint32).
 * Triangle order is not deterministic. */
kf_status kf_volume_extract_mesh(const kf_volume* vol, float* d_tris, uint32_t max_tris, uint32_t* d_count,
                                 kf_stream s);

/* ------------------------------------------------------------------------ */
/* Depth preprocessing: uint16 mm depth -> raylen (L0), bilateral-filtered depth,
 * 3-level pyramid, camera-frame vertex and normal maps per level.  Replaces
 * CameraHandler::updateCameraData and its two kernels
 * (Source/src/CameraSupport/CameraHandler.cu:65-143). */
typedef struct kf_preprocess_params {
  float depth_scale;  /* metres per input unit (0.001 for mm) */
  float min_depth_m;
  float max_depth_m;
  int32_t bilateral_radius; /* window half-size in pixels (<= 4) */
  float sigma_space_px;
  float sigma_range_m;
  float pyramid_gate_m; /* block-average gate: |d - centre| < gate */
} kf_preprocess_params;

kf_status kf_preprocess(const kf_intrinsics* k0, const kf_preprocess_params* p,
                        const uint16_t* d_depth, kf_frame_maps* live, kf_stream s);

/* Camera-side depth conditioning (optional, ahead of kf_preprocess; in != out).
 * kf_depth_median replaces d_MedianFilter (Source/src/CameraSupport/CameraAbstract.cu:100-124):
 * 5x5 median of the non-null neighbours, null if at most 12 are valid.
 * kf_depth_undistort replaces d_undistort (CameraAbstract.cu:160-221): Brown-Conrady
 * remap with dist = {k1, k2, p1, p2}, bilinear, null unless all 4 sources are valid. */
kf_status kf_depth_median(const uint16_t* d_in, uint16_t* d_out, int32_t width, int32_t height,
                          uint16_t null_value, kf_stream s);
kf_status kf_depth_undistort(const uint16_t* d_in, uint16_t* d_out, const kf_intrinsics* k, const float dist[4],
                             kf_stream s);

/* ------------------------------------------------------------------------ */
/* TSDF integration sweep.  Replaces VolumeIntegrator::Integrate / d_integrateVolume
 * (Source/src/VolumeIntegrator.cu:86-201).  A voxel is updated iff its centre
 * projects (round-half-up) into [2,W-2)x[2,H-2), its camera z is in
 * [min_depth, max_depth], the pixel's raylen is valid and sdf >= -T.
 * d_updated (nullable) receives += number of updated voxels (uint64);
 * d_update_mask (nullable, n^3/32 uint32 words, caller-zeroed) gets one bit per
 * updated voxel (bit (idx & 31) of word idx >> 5). */
typedef struct kf_integrate_params {
  float min_depth_m;
  float max_depth_m;
} kf_integrate_params;

kf_status kf_integrate(kf_volume* vol, const kf_intrinsics* k0, const kf_integrate_params* p,
                       const float* d_raylen, const kf_pose* d_pose,
                       unsigned long long* d_updated, uint32_t* d_update_mask, kf_stream s);

/* ------------------------------------------------------------------------ */
/* Raycast.  Replaces Raycaster::Raycast / d_raycast (Source/src/Raycaster.cu:97-242)
 * with trilinear sampling, linear zero-crossing refinement and trilinear
 * central-difference gradient normals.  Writes world-frame vertex/normal maps of
 * level 0 and subsamples (x2) into the coarser levels of `model`.
 * d_steps (nullable) receives += total march steps over all rays (uint64). */
typedef struct kf_raycast_params {
  float min_depth_m;  /* rays start at this camera-z depth */
  float step_far;     /* step (in units of T) while the sample is +1 (free space) */
  float step_near;    /* step (in voxels) inside the truncation band */
  int32_t max_steps;
} kf_raycast_params;

kf_status kf_raycast(const kf_volume* vol, const kf_intrinsics* k0, const kf_raycast_params* p,
                     const kf_pose* d_pose, kf_frame_maps* model,
                     unsigned long long* d_steps, kf_stream s);

/* Shaded view of the model maps (the reference's render output,
 * Source/src/Raycaster.cu:214-228): mode 0 = grey 0.6 * dot(-ray, n) + 0.2 (0 when
 * |dot| < 1e-6), mode 1 = normal map (n + 1) / 2; channels clamped and truncated to
 * bytes (R in the low byte), alpha 0, as the reference packs them.  An invalid model
 * normal counts as the zero normal of a ray without a surface (as there). */
kf_status kf_render_shaded(const kf_intrinsics* k0, const kf_frame_maps* model, const kf_pose* d_pose,
                           int32_t mode, uint32_t* d_rgba, kf_stream s);

/* ------------------------------------------------------------------------ */
/* ICP tracker.  Replaces ICP::Iterate_ICP, ICP::FindCorresponding and
 * ICP::BuildNewTransformMatrix (Source/src/ICP.cpp:84-182, Source/src/ICP.cu:116-340).
 * Projective association model->live, point-to-plane rows A=[m x d, m],
 * b = m.(s-d); per-block partial sums of the 21+6 normal-equation terms plus
 * sum b^2, inlier and candidate counts, written as one slot per block.  Each
 * iteration is one launch whose blocks all start by summing the previous
 * iteration's slots in FP64 (same order in every block), solving by FP64 LDL^T
 * and composing the Euler-ZYX increment T <- dT * T in FP64; a final one-block
 * launch solves the last iteration.  The pose never returns to the host. */
typedef struct kf_icp_params {
  int32_t levels;                     /* 1..3 */
  int32_t iterations[KF_MAX_LEVELS];  /* per level, [0] = finest; run coarse -> fine */
  float dist_thresh_m;
  float normal_thresh_deg;
  int32_t compensated;                /* 1: terms accumulated in FP64 (exact products of the FP32 row
                                         entries), block partials in FP64 (default); 0: plain FP32
                                         sums within a block */
  int32_t single_launch;              /* 1: the whole call is one launch, iterations separated by a
                                         grid barrier (same results as the multi-launch form, bit for
                                         bit, while the barrier works); 0: one launch per iteration
                                         (default).  The barrier's wait is bounded: if it times out
                                         (the device is shared with other work that keeps blocks from
                                         being co-resident), the call returns the guess with status 2,
                                         and so does every later single-launch call of the tracker
                                         until kf_tracker_reset (kf_pipeline_reset calls it).
                                         Single-launch calls that overlap on one device (several
                                         trackers, several streams) need all their blocks resident
                                         together, one per compute unit: ceil(pixels / 1536) per call
                                         up to 196,608 pixels at the finest level (320x240: 50), up to
                                         256 beyond, where such calls must not overlap. */
} kf_icp_params;

/* Per-call tracking statistics (device struct; read back with kf_memcpy_dtoh). */
typedef struct kf_icp_stats {
  int32_t status;        /* 0 ok; 1 a system was singular (pose of that iteration kept, later iterations
                            skipped); 2 the single-launch barrier timed out (the guess is returned) */
  int32_t iterations;    /* iterations that produced an update */
  int32_t inliers;       /* associations in the last executed iteration */
  int32_t candidates;    /* pixels with valid model vertex/normal and live depth, last iteration */
  double residual_rms;   /* sqrt(sum b^2 / inliers), last executed iteration (m) */
  double level_residual[KF_MAX_LEVELS];
  int32_t level_inliers[KF_MAX_LEVELS];
  int32_t skip;          /* input flag: when nonzero the call does nothing (device-side gating) */
  int32_t pad_;
} kf_icp_stats;

typedef struct kf_tracker kf_tracker;

kf_status kf_tracker_create(const kf_intrinsics* k0, const kf_icp_params* p, kf_tracker** out);
kf_status kf_tracker_destroy(kf_tracker* t);
/* Clears the tracker's control block (the single-launch form's barrier words and
 * its timed-out flag, see kf_icp_params.single_launch) on stream s. */
kf_status kf_tracker_reset(kf_tracker* t, kf_stream s);
/* Bound of each single-launch barrier wait, in polls (0: the default, about a
 * second; 1: a block that is not the last to arrive gives up at its first check).
 * Small values force the timeout path (status 2) for tests; kf_tracker_reset
 * restores the default.  Blocking. */
kf_status kf_tracker_set_barrier_polls(kf_tracker* t, uint32_t polls, kf_stream s);
/* Tracks `live` against `model` starting at *d_guess; writes the result to *d_out
 * (may alias d_guess).  d_stats (device, nullable): written with the call's stats;
 * if d_stats->skip is nonzero at execution time, the call leaves *d_out and *d_stats
 * untouched (its iteration launches still run unless the tracker's parameters ask
 * for the single-launch form, where a skipped call costs one short launch). */
kf_status kf_icp_track(kf_tracker* t, const kf_frame_maps* live, const kf_frame_maps* model,
                       const kf_pose* d_guess, kf_pose* d_out, kf_icp_stats* d_stats, kf_stream s);

/* Tracking without a tracker handle and without allocating (no counterpart in the
 * reference: for callers that cannot call hipMalloc — code under HIP graph
 * capture, tight serving loops, harnesses that forbid allocation).  The same
 * computation as kf_icp_track on a tracker created with (k0, p), bit for bit; the
 * tracker's scratch (block slots, control block, step poses, statistics) is a
 * fixed device array of the library of about 257 KiB per GPU, held until the
 * process ends.  It has slots for KF_ICP_NOALLOC_MAX_SLOTS blocks, i.e. level-0
 * images of up to 786,432 pixels (262,144 at a coarser level, where level 0 has no
 * iterations); larger images are rejected with KF_ERR_INVALID_ARGUMENT.  Every call on one GPU shares that GPU's array: calls
 * that overlap on one GPU (two streams, two host threads) race. */
#define KF_ICP_NOALLOC_MAX_SLOTS 512
kf_status kf_icp_track_noalloc(const kf_intrinsics* k0, const kf_icp_params* p, const kf_frame_maps* live,
                               const kf_frame_maps* model, const kf_pose* d_guess, kf_pose* d_out,
                               kf_icp_stats* d_stats, kf_stream s);

/* One association + reduction pass at `level` with pose *d_est (no solve);
 * writes the 30 FP64 sums {AtA upper 21 (row-major i<=j), Atb 6, sum b^2,
 * inliers, candidates} to d_sums (device, 30 doubles) and, if d_inlier_mask is
 * not NULL, one byte per model pixel (1 = associated).  For testing and tools. */
kf_status kf_icp_reduce(kf_tracker* t, int32_t level, const kf_frame_maps* live,
                        const kf_frame_maps* model, const kf_pose* d_est,
                        double* d_sums, uint8_t* d_inlier_mask, kf_stream s);

/* Constant-velocity guess on the device: T_guess = T1 * (T0^-1 * T1), FP64.
 * (prev2 = frame k-2, prev1 = frame k-1.) */
kf_status kf_pose_constant_velocity(const kf_pose* d_prev2, const kf_pose* d_prev1,
                                    kf_pose* d_guess, kf_stream s);

/* ------------------------------------------------------------------------ */
/* Learned pose prior (no counterpart in the reference, whose ICP starts from the
 * previous pose, Source/src/ICP.cpp:94).  A CNN reads two consecutive 160x120
 * depth maps (metres, 0 = invalid) and the previous frame's motion and predicts
 * the current frame's motion, which warm-starts ICP.
 *   conv 3x3/s2 2->32, 32->64, 64->64, 64->128 (ReLU) -> global average pool ->
 *   concat(previous twist) -> FC 134->256 (ReLU) -> FC 256->6 -> + previous twist.
 * Every product is a hand-written BF16 MFMA GEMM (FP32 accumulate); weights are
 * FP32 masters with BF16 copies; training is Adam on the device.
 * Twist: (w, t) with R = exp([w]x) (rotation vector) and t the translation of the
 * motion D = T_prev^-1 T_cur, scaled by 1/KF_PRIOR_ROT_SCALE and 1/KF_PRIOR_TRANS_SCALE.
 * Parameter blob (FP32): per layer W (row = output channel; conv columns ordered
 * (ky, kx, cin)) then b, for conv1..conv4, fc1, fc2. */
#define KF_PRIOR_WIDTH 160
#define KF_PRIOR_HEIGHT 120
#define KF_PRIOR_ROT_SCALE 0.05   /* rad  */
#define KF_PRIOR_TRANS_SCALE 0.05 /* metre */

typedef struct kf_prior kf_prior;

int64_t kf_prior_param_count(void);
kf_status kf_prior_create(int32_t max_batch, kf_prior** out);
kf_status kf_prior_destroy(kf_prior* p);
kf_status kf_prior_init_params(kf_prior* p, uint64_t seed); /* He-uniform init, zero biases; resets Adam */
kf_status kf_prior_set_params(kf_prior* p, const float* h_params, int64_t count); /* blocking */
kf_status kf_prior_get_params(kf_prior* p, float* h_params, int64_t count);       /* blocking */
/* Batched forward.  d_frames: [F][120][160] float depth maps; d_pairs: [batch][2]
 * int32 frame indices (previous, current); d_prev_twist, d_out: [batch][6] scaled twists. */
kf_status kf_prior_forward(kf_prior* p, const float* d_frames, const int32_t* d_pairs, const float* d_prev_twist,
                           int32_t batch, float* d_out, kf_stream s);
/* Forward + backward of the loss mean((out - target)^2) over batch*6 outputs;
 * writes dLoss/dparams (FP32, param_count) to d_grad and the loss to d_loss (nullable). */
kf_status kf_prior_gradients(kf_prior* p, const float* d_frames, const int32_t* d_pairs, const float* d_prev_twist,
                             const float* d_target, int32_t batch, float* d_grad, float* d_loss, kf_stream s);
/* One Adam step (beta1 0.9, beta2 0.999, eps 1e-8) on that loss; d_loss nullable. */
kf_status kf_prior_train_step(kf_prior* p, const float* d_frames, const int32_t* d_pairs,
                              const float* d_prev_twist, const float* d_target, int32_t batch, float lr,
                              float* d_loss, kf_stream s);

/* ------------------------------------------------------------------------ */
/* Frame pipeline: the per-frame driver of RunApp::display
 * (Source/src/MainApp.cpp:774-970) in KinectFusion order
 * preprocess -> ICP (guess: constant velocity or learned prior) -> integrate -> raycast,
 * recorded once into a hipGraph and replayed per frame. */
typedef struct kf_pipeline_desc {
  kf_intrinsics intr;
  kf_volume_desc volume;
  kf_preprocess_params pre;
  kf_integrate_params integ;
  kf_raycast_params ray;
  kf_icp_params icp;          /* plain ICP (from the constant-velocity guess) */
  kf_icp_params icp_prior;    /* warm-started ICP used when a prior is attached */
  float fallback_residual_ratio; /* prior fallback: residual > ratio * running median */
  float fallback_min_inlier_frac; /* prior fallback: inliers / candidates below this */
  int32_t use_graph;          /* 1: record and replay a hipGraph per frame */
} kf_pipeline_desc;

typedef struct kf_frame_stats {
  int32_t frame;
  int32_t used_prior;   /* the learned prior supplied the guess */
  int32_t fell_back;    /* prior result rejected; plain ICP result used */
  int32_t pad_;
  kf_icp_stats icp;          /* ICP that produced the pose */
  kf_icp_stats icp_prior;    /* warm-started ICP (valid if used_prior) */
  unsigned long long updated_voxels; /* stage-timing mode only: voxels updated by the sweep */
  unsigned long long raycast_steps;  /* stage-timing mode only: total march steps */
  int32_t prior_frames;      /* frames tracked with the prior since the last reset */
  int32_t prior_fallbacks;   /* of which fell back to plain ICP */
} kf_frame_stats;

typedef struct kf_pipeline kf_pipeline;

kf_status kf_pipeline_default_desc(kf_pipeline_desc* d);
/* s = NULL: the pipeline creates (and owns) a non-blocking stream of its own. */
kf_status kf_pipeline_create(const kf_pipeline_desc* d, kf_stream s, kf_pipeline** out);
kf_status kf_pipeline_destroy(kf_pipeline* p);
/* Clears the volume, sets frame 0's pose (host T_wc) and the frame counter. */
kf_status kf_pipeline_reset(kf_pipeline* p, const double T0_wc[16]);
/* Processes one uint16 depth frame already in device memory (asynchronous on the
 * pipeline stream).  As in RunApp::display (Source/src/MainApp.cpp:774-970), a call
 * first integrates and raycasts the previous frame, then tracks this one: the pose
 * of this frame is available when the call's work completes, its integration into
 * the volume follows at the start of the next call (kf_pipeline_flush, which the
 * volume and map accessors call, does it at once).  With a prior attached, the
 * previous frame's integration and raycast run concurrently with this frame's
 * preprocessing and prior inference (a second stream of the pipeline's own). */
kf_status kf_pipeline_process(kf_pipeline* p, const uint16_t* d_depth);
/* The same with the frame in pinned host memory (kf_host_malloc_pinned /
 * hipHostMalloc; anything else is rejected with KF_ERR_INVALID_ARGUMENT), as
 * CameraAbstract::GetDepthFrame hands over a host frame that the reference uploads
 * inside its frame (Source/src/CameraSupport/CameraFromFile.cpp:84-86).  The
 * frame's first kernel reads the caller's buffer over the bus into the pipeline's
 * staging buffer (with a prior attached, while the previous frame's integration and
 * raycast run), so the upload is part of the frame.  Both forms require a 16-byte
 * aligned frame, and the buffer must stay unchanged until the frame's work has run
 * (kf_pipeline_get_pose, or the pipeline stream synchronised). */
kf_status kf_pipeline_process_host(kf_pipeline* p, const uint16_t* h_depth);
/* Integrates and raycasts the last tracked frame now if that is still pending. */
kf_status kf_pipeline_flush(kf_pipeline* p);
/* Attaches a learned prior (not owned; NULL detaches) before the next tracked frame.
 * Each frame then: prior guess -> ICP with icp_prior iterations -> accept, or fall
 * back to plain ICP from the constant-velocity guess when that ICP failed, its
 * residual exceeds fallback_residual_ratio x the running median of the last 31
 * accepted residuals, or its inliers / candidates < fallback_min_inlier_frac.
 * Requires a 640x480 level 0 with 3 levels (the prior reads the 160x120 level). */
kf_status kf_pipeline_attach_prior(kf_pipeline* p, kf_prior* prior);
kf_status kf_pipeline_get_pose(kf_pipeline* p, double T_wc[16]);          /* blocking */
/* Poses of every frame since the last reset (device log, up to KF_TRAJ_CAPACITY
 * frames, written by the pipeline itself): copies min(frames, max_frames) T_wc
 * into T_out (host, 16 doubles each) and the logged frame count into *frames. */
#define KF_TRAJ_CAPACITY 8192
kf_status kf_pipeline_get_trajectory(kf_pipeline* p, double* T_out, int32_t max_frames,
                                     int32_t* frames); /* blocking */
kf_status kf_pipeline_get_stats(kf_pipeline* p, kf_frame_stats* stats);   /* blocking */
/* Both flush first: the volume holds every processed frame, the model maps are the
 * raycast at the last pose, the live maps those of the last frame. */
kf_status kf_pipeline_get_volume(kf_pipeline* p, kf_volume** vol);
kf_status kf_pipeline_get_maps(kf_pipeline* p, kf_frame_maps* live, kf_frame_maps* model);
kf_status kf_pipeline_get_stream(kf_pipeline* p, kf_stream* s);
/* Stage-timing mode (eager launches, hipEvents on the pipeline stream, voxel and
 * march-step counters; frames are processed in order without deferral or overlap).
 * Times (ms) of the last processed frame:
 * [preprocess, guess+icp, raylen tiles + brick classes, sweep kernel, brick
 *  distances, raycast kernel (with the model pyramid), pose log]; the sweep and
 * raycast entries are the kernels' own start-to-end times, the others the time
 * between events around the stage. */
#define KF_STAGES 7
kf_status kf_pipeline_set_stage_timing(kf_pipeline* p, int32_t on);
/* Stage-timing counters of the last frame: [voxels updated by the sweep, raycast
 * march steps, raycast samples that loaded their eight corners, raycast sample
 * batches (per lane), raycast steps taken by the free-space skip, sum over
 * wavefronts of 64 x the largest batch count of their rays, the largest batch
 * count of any ray]. */
#define KF_COUNTERS 7
kf_status kf_pipeline_get_counters(kf_pipeline* p, uint64_t out[KF_COUNTERS]);
kf_status kf_pipeline_get_stage_ms(kf_pipeline* p, float ms[KF_STAGES]);

#ifdef __cplusplus
}
#endif

#endif /* KINFU_H_ */
