#!/usr/bin/env python3
"""Headline benchmark of the KinectFusion hot path on one MI355X.

Workload: the seeded 300-frame 640x480 synthetic stream (3x3x3 m room, 6-10
random primitives, smooth path <= 3 cm / 2 deg per frame), tracked and fused into
a 512^3 volume over a 4 m cube (T = 0.02 m).  A step is one frame: upload of the
uint16 depth frame from pinned host memory (read by the frame's first kernel) ->
bilateral + pyramid + vertex/normal maps -> 3-level ICP (10/5/4 iterations, FP64
solve on the device) -> TSDF sweep -> raycast.  Frames 0..W-1 warm up, frames
W..W+K-1 are timed.  The scene and trajectory are those of the full 300-frame
stream whatever W + K is (a shorter run times a prefix of it).

Variants on the same stream: plain FP32 volume (8 B/voxel), packed FP16+u16
volume (4 B/voxel), and FP16 + the learned pose prior (ICP warm-started with
4/3/3 iterations, plain 10/5/4 fallback) when trained weights are present;
`value` is the fps of the last of these that ran (learned + FP16 normally), with
the upload inside the frame; each variant is also timed with the frames already
in HBM (`fps_frames_in_hbm`) for comparison.  A
stage-timing pass (hipEvents on the pipeline's stream around each kernel group)
gives per-kernel times; with the kernels' algorithmic bytes (sweep U*2*B_v + P*4
with U from the sweep's own update counter, raycast P*(S*B_t + 24) with S from its
step counter, ICP sum over iterations of P_l*49 + partial slots) they give achieved
GB/s and the fraction of the 8 TB/s HBM peak per kernel; `roofline` is the longer
of the sweep and the raycast.  `traffic` comes from the committed rocprofv3
FETCH_SIZE / WRITE_SIZE summary of the same workload.  The CPU baseline runs the
oracle (OpenMP restatement of the reference's per-voxel / per-pixel bodies) on a
bounded sample of the FP32 stream on the host cores; in the same leg the oracle's
FP64 instantiation checks the FP16 pipeline's accuracy (TSDF, raycast depth, pose
drift) on the first frames, reported as `accuracy`.

Prints ONE JSON line.  `--gpus N` with N > 1 is not supported (one GPU).
"""
from __future__ import annotations

import argparse
import json
import os
import platform
import statistics
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "fps (ICP+integrate+raycast) 512³/640×480, learned+FP16 vs plain; ATE mm"
HBM_PEAK_GBS = 8000.0


def log(msg: str) -> None:
    print(msg, file=sys.stderr, flush=True)


def cpu_model() -> str:
    try:
        for ln in open("/proc/cpuinfo"):
            if ln.startswith("model name"):
                return ln.split(":", 1)[1].strip()
    except OSError:
        pass
    return platform.processor() or "unknown"


def attach_prior(kf, p):
    from openfusion_amd import prior_train
    prior = kf.Prior(max_batch=1)
    prior_train.load(prior, prior_train.DEFAULT_WEIGHTS)
    p.attach_prior(prior)
    return prior


def timed_run(kf, synth, metrics, stream, frames_src, preset: str, W: int, K: int, use_prior: bool = False,
              host: bool = True) -> dict:
    """W warm-up frames, then K timed frames.  host: each frame is handed over in
    pinned host memory (kf_pipeline_process_host; its upload is part of the frame),
    else already in device memory (kf_pipeline_process)."""
    import ctypes as C
    desc = synth.pipeline_desc(preset)
    p = kf.Pipeline(desc)
    if use_prior:
        attach_prior(kf, p)
    fb = stream.depth[0].nbytes
    feed = (lambda i: p.process_host(frames_src.ptr + i * fb)) if host else \
        (lambda i: p.process(frames_src.ptr + i * fb))
    p.reset(stream.poses[0])
    for i in range(W):
        feed(i)
    kf.synchronize()
    s = p.stream()
    L = kf.lib()
    e0, e1 = C.c_void_p(), C.c_void_p()
    kf.check(L.kf_event_create(C.byref(e0)), "event")
    kf.check(L.kf_event_create(C.byref(e1)), "event")
    kf.check(L.kf_event_record(e0, s), "record")
    t0 = time.perf_counter()
    for i in range(W, W + K):
        feed(i)
    kf.check(L.kf_event_record(e1, s), "record")
    kf.synchronize()
    wall = time.perf_counter() - t0
    ms = C.c_float()
    kf.check(L.kf_event_elapsed_ms(e0, e1, C.byref(ms)), "elapsed")
    L.kf_event_destroy(e0)
    L.kf_event_destroy(e1)
    traj = p.trajectory()
    n = min(traj.shape[0], W + K)
    st = p.stats()
    p.close()
    extra = {}
    if use_prior:
        extra = {"prior_frames": int(st.prior_frames), "prior_fallbacks": int(st.prior_fallbacks),
                 "fallback_rate": float(st.prior_fallbacks) / max(1, st.prior_frames)}
    return {
        **extra,
        "fps": K / wall,
        "ms_per_frame": 1000.0 * wall / K,
        "gpu_ms_per_frame": ms.value / K,
        "ate_mm": 1000.0 * metrics.ate(traj[:n], stream.poses[:n]),
        "ate_aligned_mm": 1000.0 * metrics.ate_aligned(traj[:n], stream.poses[:n]),
        "last_inliers": int(st.icp.inliers),
        "last_iterations": int(st.icp.iterations),
    }


def stage_run(kf, synth, stream, dd, preset: str, W: int, S: int, use_prior: bool = False) -> dict:
    desc = synth.pipeline_desc(preset)
    p = kf.Pipeline(desc)
    if use_prior:
        attach_prior(kf, p)
    p.set_stage_timing(True)
    fb = stream.depth[0].nbytes
    p.reset(stream.poses[0])
    rows = []
    for i in range(W + S):
        p.process(dd.ptr + i * fb)
        if i >= W:
            st = p.stats()
            rows.append((p.stage_ms(), st.updated_voxels, st.raycast_steps, p.counters()))
    vstats = p.volume().stats()  # one full read of the volume (also a known-size read for counters)
    p.close()
    ms = np.array([r[0] for r in rows])
    U = np.array([r[1] for r in rows], dtype=np.float64)
    steps = np.array([r[2] for r in rows], dtype=np.float64)
    cnt = np.array([r[3] for r in rows], dtype=np.float64)
    return {"ms": ms, "U": U, "steps": steps, "counters": cnt, "desc": desc, "observed_voxels": float(vstats[0])}


def kernel_rooflines(kf, d, sr: dict, prior: bool) -> dict:
    """Algorithmic bytes per launch / average launch time for the sweep, the raycast
    and ICP (per frame), from the stage-timing run (hipEvents on the pipeline stream)."""
    P = d.intr.width * d.intr.height
    n = d.volume.n
    Bv = 4 if d.volume.format == kf.KF_VOXEL_F16 else 8
    ms = sr["ms"]
    out = {}
    sweep_bytes = float((sr["U"] * 2 * Bv + P * 4).mean())
    t = float(ms[:, 3].mean())
    out["integrate"] = {"kernel": f"integrate<{'FP16' if Bv == 4 else 'FP32'}> (TSDF sweep)",
                        "algorithmic_bytes": sweep_bytes, "avg_launch_ms": t,
                        "updated_voxels_per_launch": float(sr["U"].mean()),
                        "upper_bound_bytes": float(n ** 3 * 2 * Bv + P * 4)}
    S_bar = float(sr["steps"].mean() / P)
    ray_bytes = P * (S_bar * (Bv // 2) + 24)
    t = float(ms[:, 5].mean())
    c = sr["counters"].mean(0)
    out["raycast"] = {"kernel": f"raycast<{'FP16' if Bv == 4 else 'FP32'}>", "algorithmic_bytes": ray_bytes,
                      "avg_launch_ms": t, "mean_steps_per_ray": S_bar,
                      "per_ray": {"samples_loading_corners": round(float(c[2]) / P, 2),
                                  "sample_batches": round(float(c[3]) / P, 2),
                                  "steps_skipped_in_free_space": round(float(c[4]) / P, 2),
                                  "batches_of_the_longest_ray_per_wave": round(float(c[5]) / P, 2),
                                  "batches_of_the_longest_ray": round(float(sr["counters"][:, 6].max()), 2)}}
    icp = d.icp_prior if prior else d.icp
    icp_bytes = 0.0
    for lvl in range(icp.levels):
        Pl = P >> (2 * lvl)
        per = next((p for p in (256, 512, 1280) if Pl <= 256 * p), 1536)  # pixels of a step's block
        blocks = min(1024, -(-Pl // per))
        icp_bytes += icp.iterations[lvl] * (Pl * 49 + 2 * blocks * 256)
    t = float(ms[:, 1].mean())
    out["icp"] = {"kernel": "guess + icp_step (per frame, "
                            f"{'/'.join(str(icp.iterations[i]) for i in range(icp.levels))} iterations)",
                  "algorithmic_bytes": icp_bytes, "avg_launch_ms": t}
    for k in out.values():
        k["achieved_GBs"] = round(k["algorithmic_bytes"] / (k["avg_launch_ms"] * 1e-3) / 1e9, 1)
        k["frac"] = round(k["achieved_GBs"] / HBM_PEAK_GBS, 4)
    return out


TRAFFIC_FILES = {"full": "traffic_512_full.json", "stress": "traffic_768_stress.json"}


def profiled_traffic(kernel: str, Bv: int, workload: str) -> dict | None:
    """HBM bytes per dispatch of the kernel (its FP16 or FP32 instantiation) from the
    committed rocprofv3 FETCH_SIZE / WRITE_SIZE summary of this workload, scaled by
    the calibration kernels; None when the summary or the kernel is missing."""
    name = TRAFFIC_FILES[workload]
    try:
        with open(os.path.join(ROOT, "profiles", name)) as f:
            t = json.load(f)
    except (OSError, ValueError):
        return None
    prefix = f"{kernel}<{1 if Bv == 4 else 0}"
    hits = [(key, k) for key, k in t.get("kernels", {}).items() if k["kernel"].startswith(prefix)]
    if not hits:
        return None
    key, k = max(hits, key=lambda h: h[1]["dispatches"])
    return {"bytes": k["fetch_bytes"] + k["write_bytes"], "source": f"profiles/{name}[{key}]"}


def cpu_baseline(orc, synth, stream, preset: str, frames: int) -> dict:
    desc = synth.pipeline_desc(preset)
    p = orc.Pipeline(desc, 0)
    p.reset(stream.poses[0])
    totals, stages = [], []
    t0 = time.perf_counter()
    for i in range(frames):
        p.process(stream.depth[i])
        if i >= 2:  # frame 0 has no ICP; frame 1 warms caches
            ms = p.stage_ms()
            stages.append(ms)
            totals.append(float(ms.sum()))
    wall = time.perf_counter() - t0
    med = statistics.median(totals)
    return {"fps": 1000.0 / med, "median_frame_ms": med, "stage_ms": np.median(np.array(stages), 0).tolist(),
            "wall_s": wall, "threads": orc.num_threads(), "frames": frames}


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=290, help="timed frames")
    ap.add_argument("--warmup", type=int, default=10, help="untimed frames (steady state starts at 10)")
    ap.add_argument("--stage-frames", type=int, default=40)
    ap.add_argument("--cpu-frames", type=int, default=8, help="frames of the bounded CPU baseline sample")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-hbm", action="store_true", help="skip the comparison runs with frames already in HBM")
    ap.add_argument("--accuracy-frames", type=int, default=8,
                    help="frames of the FP16-vs-FP64-oracle accuracy check in the CPU-baseline leg (0: skip)")
    ap.add_argument("--only", choices=["plain", "fp16", "learned_fp16"], default=None)
    ap.add_argument("--no-prior", action="store_true", help="skip the learned-prior variant")
    ap.add_argument("--workload", choices=["full", "stress"], default="full",
                    help="full: 512^3 / 4 m, 300 frames (headline); stress: 768^3 / 6 m, 1000 frames with bursts")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py: --gpus {args.gpus} is not supported: this build runs on one GPU "
              "(the sharded volume design is documented, not built).", file=sys.stderr)
        return 2

    from openfusion_amd import kinfu as kf, metrics, synth
    if kf.device_count() < 1:
        print("bench.py: no GPU visible", file=sys.stderr)
        return 1
    W, K = args.warmup, args.steps
    stress = args.workload == "stress"
    if stress and K == 290:
        K = 990
    frames = W + K
    P32, P16 = ("stress32", "stress") if stress else ("full", "full16")
    t = time.perf_counter()
    stream = synth.make_stream(P16 if stress else "full", frames=max(frames, W + args.stage_frames, args.cpu_frames))
    scene_id = f"{stream.scene.count} primitives, digest {synth.scene_digest(stream.scene)}"
    log(f"stream: {stream.depth.shape[0]} frames, {scene_id} ({time.perf_counter()-t:.1f}s)")
    dd = kf.upload(stream.depth)  # device copy: in-HBM comparison runs and the stage-timing pass
    pinned = kf.PinnedBuffer(stream.depth.nbytes)  # the frames as a camera driver hands them over
    pinned.view(np.uint16, stream.depth.shape)[...] = stream.depth

    from openfusion_amd import prior_train
    have_prior = os.path.exists(prior_train.DEFAULT_WEIGHTS) and not args.no_prior
    variants = [("plain", P32, False), ("fp16", P16, False)]
    if have_prior:
        variants.append(("learned_fp16", P16, True))
    res = {}
    for name, preset, use_prior in variants:
        if args.only and args.only != name:
            continue
        log(f"timed run {name} ({preset}{' + prior' if use_prior else ''}): warmup {W}, steps {K}, "
            "frames from pinned host memory")
        res[name] = timed_run(kf, synth, metrics, stream, pinned, preset, W, K, use_prior, host=True)
        log(f"  {name}: {res[name]['fps']:.1f} fps, ATE {res[name]['ate_mm']:.3f} mm")
        if not args.no_hbm:
            r = timed_run(kf, synth, metrics, stream, dd, preset, W, K, use_prior, host=False)
            res[name]["fps_frames_in_hbm"] = r["fps"]
            log(f"  {name} (frames already in HBM): {r['fps']:.1f} fps")

    head = "learned_fp16" if "learned_fp16" in res else ("fp16" if "fp16" in res else "plain")
    head_preset = P32 if head == "plain" else P16
    head_prior = head == "learned_fp16"
    log(f"stage timing ({head}, {args.stage_frames} frames)")
    sr = stage_run(kf, synth, stream, dd, head_preset, W, args.stage_frames, head_prior)
    d = sr["desc"]
    n = d.volume.n
    Bv = 4 if d.volume.format == kf.KF_VOXEL_F16 else 8
    P = d.intr.width * d.intr.height
    stage = sr["ms"].mean(0)
    kernels = kernel_rooflines(kf, d, sr, head_prior)
    dominant = max(("integrate", "raycast"), key=lambda k: kernels[k]["avg_launch_ms"])
    dom = kernels[dominant]
    traffic = profiled_traffic(dominant, Bv, args.workload)
    pre = synth.PRESETS[head_preset]

    out = {
        "metric": METRIC,
        "value": round(res[head]["fps"], 2),
        "unit": "fps",
        "n_gpus": 1,
        "steps": K,
        "warmup": W,
        "ms_per_step": round(res[head]["ms_per_frame"], 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic",
        "config": {
            "workload": f"{n}^3 {'FP16+u16' if Bv == 4 else 'FP32+FP32'} TSDF over {pre.extent:g} m "
                        f"(T {pre.trunc:g} m), 640x480, seeded {stream.depth.shape[0]}-frame synthetic stream "
                        f"({'bursts up to 6 cm / 5 deg' if stress else '<= 3 cm / 2 deg'} per frame), ICP 3 levels "
                        + ("4/3/3 warm-started by the learned prior (fallback: plain 10/5/4)" if head_prior else
                           "10/5/4 from the constant-velocity guess"),
            "volume_format": "f16+u16" if Bv == 4 else "f32+f32",
            "frames_timed": f"{W}..{W + K - 1}",
            "frames_from": "pinned host memory (upload inside the frame)",
            "scene": scene_id,
            "variant": head,
        },
        "roofline": {
            "kernel": dom["kernel"],
            "bound": "hbm",
            "achieved": dom["achieved_GBs"],
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": round(dom["achieved_GBs"] / HBM_PEAK_GBS, 4),
            "traffic": traffic["bytes"] if traffic else None,
            "traffic_source": traffic["source"] if traffic else None,
            "algorithmic_bytes_per_launch": dom["algorithmic_bytes"],
            "avg_launch_ms": dom["avg_launch_ms"],
        },
        "kernels": kernels,
        "variants": {k: {kk: (round(vv, 4) if isinstance(vv, float) else vv) for kk, vv in v.items()}
                     for k, v in res.items()},
        "observed_voxels_after_stage_run": sr["observed_voxels"],
        "stages_ms": dict(zip(["preprocess", "guess+icp", "brick_classes", "sweep", "brick_distances", "raycast",
                               "pose_log"],
                              [round(float(x), 4) for x in stage])),
    }
    if "plain" in res:
        for name in ("fp16", "learned_fp16"):
            if name in res:
                out[f"speedup_{name}_vs_plain"] = round(res[name]["fps"] / res["plain"]["fps"], 3)
        out["ate_mm"] = round(res[head]["ate_mm"], 3)
        out["ate_plain_mm"] = round(res["plain"]["ate_mm"], 3)
    if not args.no_cpu:
        # CPU-baseline leg: the oracle runs here as the baseline and as the checker of
        # the accuracy block, never as the thing measured.
        from oracle import oracle as orc
        log(f"cpu baseline: oracle FP32 pipeline, {args.cpu_frames} frames at {n}^3")
        cb = cpu_baseline(orc, synth, stream, P32, args.cpu_frames)
        out["cpu_baseline"] = {
            "value": round(cb["fps"], 3), "unit": "fps", "cores": cb["threads"], "kind": "port",
            "sample": f"frames 2..{args.cpu_frames - 1} of the {n}^3 FP32 stream (median per-frame time of "
                      f"preprocess+ICP+integrate+raycast; frames 0-1 warm-up), {cpu_model()}",
            "stage_ms": [round(x, 2) for x in cb["stage_ms"]],
        }
        if args.accuracy_frames > 0 and not stress:
            from oracle import accuracy
            log(f"accuracy: FP16 GPU pipeline vs FP64 oracle, {args.accuracy_frames} frames")
            a = accuracy.fp16_vs_fp64(kf, orc, synth, metrics, args.accuracy_frames)
            out["accuracy"] = {
                "vs": "FP64 oracle (FP64 maps, volume, ICP) on frames 0-%d" % (args.accuracy_frames - 1),
                "tsdf_abs_err_over_T_p999": a["tsdf_abs_err_over_T"]["p999"],
                "tsdf_abs_err_over_T_max": a["tsdf_abs_err_over_T"]["max"],
                "raycast_depth_rmse_mm": round(a["raycast_depth_rmse_mm"], 4),
                "raycast_silhouette_flips": a["raycast_silhouette_flips"],
                "pose_drift_max_mm": round(a["pose_drift_max_mm"], 4),
                "pose_drift_max_deg": round(a["pose_drift_max_deg"], 5),
            }
    print(json.dumps(out), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
