#!/usr/bin/env python3
"""Throughput of the exact phantom hair path on one MI355X.

Workload (one "step" = one frame): 100,000 seeded strands x 32 cubic Bezier segments
(3.2M segments, tapered per-point radius 0.04 -> 0.01 mm) traced with the phantom ray-hair
intersector at 1920x1080: one primary ray per pixel plus one shadow ray per hit, shaded with
Shade() x visibility into an RGBA8 image. FP32 with FP64 polish of grazing roots.

value = (primary + shadow rays per frame) / frame time, Mrays/s, scene resident in HBM.
roofline: algorithmic bytes of the dominant kernel per launch (32 B ray + 16 B hit + 64 B per
candidate segment, N*_prim counted on the GPU) / its average launch time (HIP events on the
launch stream), against 8 TB/s. cpu_baseline: the oracle (host C++ transliteration of the
reference GLSL, BVH2) on a bounded pixel sample of the same frame, all host threads.

Prints one JSON line on stdout; progress goes to stderr.
"""
import argparse
import json
import math
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "Mrays/s, 100k-strand 1080p primary+shadow; exact vs neural shadows @PSNR>=40dB"
HBM_PEAK_GBS = 8000.0
FP32_PEAK_TFLOPS = 157.3  # MI355X dense FP32 vector
# FP32 operations of one 8-wide node test (node_visit in vkhrt_amd/csrc/trace_impl.hpp): 3 scale
# products, 3 origin differences and products, and per child slot 6 dequantizing fused
# multiply-adds (2 each) and the far-plane widening product: 3 + 6 + 8 x 13 = 113
NODE_TEST_FLOP = 113
# frozen view of the 100k-strand hair ball (fills the frame height)
CAMERA_EYE = (0.0, 60.0, 300.0)
CAMERA_TARGET = (0.0, 40.0, 0.0)


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--strands", type=int, default=100000)
    ap.add_argument("--segments", type=int, default=32)
    ap.add_argument("--width", type=int, default=1920)
    ap.add_argument("--height", type=int, default=1080)
    ap.add_argument("--seed", type=int, default=20240601)
    ap.add_argument("--polish", type=int, default=1, help="FP64 polish of grazing roots (1) or off (0)")
    ap.add_argument("--accurate", type=int, default=1,
                    help="headline frame re-evaluates every primary phantom hit in double-word FP32 (1: its normals "
                         "meet 1e-4 rad against FP64) or keeps the FP32 hits (0)")
    ap.add_argument("--stack-kind", type=int, default=1)
    ap.add_argument("--leaf-size", type=int, default=1)
    ap.add_argument("--persistent", type=int, default=1)
    ap.add_argument("--refill-min", type=int, default=16)
    ap.add_argument("--blocks-per-cu", type=int, default=0, help="persistent blocks per CU (0: occupancy limit)")
    ap.add_argument("--ray-order", type=int, default=0, help="0 row-major, 1 8x8 tiles, 2 64x64 tiles of 8x8 tiles")
    ap.add_argument("--xcd-chunk", type=int, default=4096,
                    help="rays handed out per XCD in runs of this many (0: one work counter)")
    ap.add_argument("--steps-per-iteration", type=int, default=3,
                    help="persistent phantom traversal: traversal steps per bookkeeping pass (1..8)")
    ap.add_argument("--shadow-group-lanes", type=int, default=16,
                    help="lanes per ray of the neural fallback's lane-group walker (8, 16, 32 or 64)")
    ap.add_argument("--cpu-seconds", type=float, default=12.0, help="target CPU-baseline sample time")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-roofline", action="store_true")
    ap.add_argument("--no-neural", action="store_true", help="skip the neural shadow form")
    ap.add_argument("--no-modes", action="store_true", help="skip the LSS, DOTS and voxel forms of the frame")
    ap.add_argument("--no-collapse-study", action="store_true",
                    help="skip the comparison of the greedy and SAH collapses to wide nodes")
    ap.add_argument("--voxel-size", type=float, default=0.5, help="cell edge of the voxel form")
    ap.add_argument("--no-batch", action="store_true", help="skip the batched multi-view path-traced form")
    ap.add_argument("--no-area", action="store_true", help="skip the 16M-segment area-light neural form")
    ap.add_argument("--autotune", type=int, default=1, help="pick BVH width, leaf size, stack kind, blocks per CU, "
                    "refill minimum and ray order with the autotuner before timing (1) or use the flags (0)")
    ap.add_argument("--neural-views", type=int, default=32, help="training views for the shadow MLP")
    ap.add_argument("--neural-epochs", type=int, default=80)
    ap.add_argument("--neural-thresholds", type=str, default="",
                    help="comma-separated variance thresholds of the neural sweeps (default: the fixed list)")
    ap.add_argument("--copy-calibration", type=int, default=0, metavar="MIB",
                    help="run a plain float32 copy kernel over MIB MiB three times and exit "
                         "(the known-size reference for the FETCH_SIZE / WRITE_SIZE counters)")
    args = ap.parse_args()
    if args.neural_thresholds:
        global NEURAL_THRESHOLDS
        NEURAL_THRESHOLDS = tuple(float(x) for x in args.neural_thresholds.split(","))
    if args.copy_calibration:
        copy_calibration(args.copy_calibration << 20)
        return

    world = int(os.environ.get("WORLD_SIZE", "1"))
    if args.gpus != 1 or world != 1:
        print(f"bench.py: this build measures one GPU only (asked for --gpus {args.gpus}, "
              f"WORLD_SIZE {world}); multi-GPU sharding is a design note, not a measured path",
              file=sys.stderr)
        sys.exit(2)

    import numpy as np
    import torch
    import vkhrt_amd as V

    assert torch.cuda.is_available(), "bench.py needs a GPU"
    torch.cuda.init()
    stream = torch.cuda.current_stream()
    sp = stream.cuda_stream
    ctx = V.Context(0)
    ctx.set_option(V.OPTION_STACK_KIND, args.stack_kind)
    ctx.set_option(V.OPTION_PERSISTENT, args.persistent)
    ctx.set_option(V.OPTION_REFILL_MIN, args.refill_min)
    ctx.set_option(V.OPTION_RAY_ORDER, args.ray_order)
    ctx.set_option(V.OPTION_XCD_CHUNK, args.xcd_chunk)
    ctx.set_option(V.OPTION_BLOCKS_PER_CU, args.blocks_per_cu)
    ctx.set_option(V.OPTION_SHADOW_GROUP_LANES, args.shadow_group_lanes)
    ctx.set_option(V.OPTION_STEPS_PER_ITERATION, args.steps_per_iteration)

    NS, SEG, W, H = args.strands, args.segments, args.width, args.height
    nseg_total = NS * SEG
    log(f"[bench] scene {NS} strands x {SEG} segments = {nseg_total} segments, {W}x{H}")
    verts = torch.empty(NS * (SEG + 1) * 4, dtype=torch.float32, device="cuda")
    lines = torch.empty(nseg_total * 8, dtype=torch.float32, device="cuda")
    curves = torch.empty(nseg_total * 16, dtype=torch.float32, device="cuda")
    ctx.generate_strands(args.seed, NS, SEG, verts.data_ptr(), stream=sp)
    ctx.generate_lines(verts.data_ptr(), NS, SEG, lines.data_ptr(), stream=sp)
    ctx.generate_curves(lines.data_ptr(), nseg_total, curves.data_ptr(), stream=sp)
    del verts, lines
    blas = V.BottomLevelAccelerationStructure(ctx, V.GEOMETRY_PHANTOM_CURVES, curves.data_ptr(),
                                              nseg_total, flags=V.BLAS_PER_POINT_RADIUS,
                                              leaf_size=args.leaf_size, stream=sp)
    tlas = V.TopLevelAccelerationStructure(ctx, [blas], stream=sp)
    torch.cuda.synchronize()
    binfo = blas.info()
    log(f"[bench] BLAS built: {binfo}")

    cam = V.camera_look_at(CAMERA_EYE, CAMERA_TARGET, fov_deg=60.0, aspect=W / H)
    image = torch.empty(W * H, dtype=torch.int32, device="cuda")
    base_flags = V.RENDER_SHADOWS | V.RENDER_RGBA8 | (V.RENDER_FP64_POLISH if args.polish else 0)
    flags = base_flags | (V.RENDER_ACCURATE_NORMALS if args.accurate else 0)
    tuning = None
    if args.autotune:
        t0 = time.perf_counter()
        tb = ctx.autotune_blas(V.GEOMETRY_PHANTOM_CURVES, curves.data_ptr(), nseg_total, cam, W, H, image.data_ptr(),
                               blas_flags=V.BLAS_PER_POINT_RADIUS, render_flags=flags, repeats=3, stream=sp)
        tlas.close()
        blas.close()
        blas = V.BottomLevelAccelerationStructure(ctx, V.GEOMETRY_PHANTOM_CURVES, curves.data_ptr(),
                                                  nseg_total, flags=V.BLAS_PER_POINT_RADIUS, stream=sp)
        tlas = V.TopLevelAccelerationStructure(ctx, [blas], stream=sp)
        tr = ctx.autotune_render(tlas, cam, W, H, image.data_ptr(), flags=flags, repeats=9, stream=sp)
        torch.cuda.synchronize()
        binfo = blas.info()
        tuning = {"bvh_width": tb["bvh_width"], "leaf_size": tb["leaf_size"], "bvh_collapse": tb["bvh_collapse"],
                  "stack_kind": tr["stack_kind"],
                  "blocks_per_cu": tr["blocks_per_cu"], "refill_min": tr["refill_min"], "ray_order": tr["ray_order"],
                  "xcd_chunk": tr["xcd_chunk"], "steps_per_iteration": tr["steps_per_iteration"],
                  "trials": tb["trials"] + tr["trials"], "seconds": round(time.perf_counter() - t0, 2),
                  "start_ms": round(tb["baseline_ms"], 4), "tuned_ms": round(tr["best_ms"], 4)}
        log(f"[bench] autotuned: {tuning}")

    def frame():
        ctx.render(tlas, cam, W, H, image.data_ptr(), flags=flags, stream=sp)

    for _ in range(args.warmup):
        frame()
    torch.cuda.synchronize()
    ctx.synchronize(sp)
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    t_wall0 = time.perf_counter()
    e0.record(stream)
    for _ in range(args.steps):
        frame()
    e1.record(stream)
    torch.cuda.synchronize()
    t_wall = time.perf_counter() - t_wall0
    ms = e0.elapsed_time(e1) / args.steps
    ctx.synchronize(sp)  # raises on traversal stack overflow
    n_primary, n_shadow = ctx.render_ray_counts()
    rays = n_primary + n_shadow
    mrays = rays / (ms * 1e-3) / 1e6
    log(f"[bench] {ms:.3f} ms/frame ({t_wall / args.steps * 1e3:.3f} wall), primary {n_primary}, "
        f"shadow {n_shadow}, {mrays:.1f} Mrays/s")

    # per-kernel HIP-event timing on the launch stream
    ctx.profiling(True)
    for _ in range(args.steps):
        frame()
    torch.cuda.synchronize()
    kstats = {k: ctx.kernel_stats(k) for k in ("render_primary", "render_shadow")}
    ctx.profiling(False)
    kavg = {k: (v[0] / v[1] if v[1] else 0.0) for k, v in kstats.items()}
    log(f"[bench] kernel avg ms: {kavg}")

    # the other form of the frame: FP32 hits only (normals miss the 1e-4 rad bound against FP64),
    # or, when the headline keeps FP32 hits, the double-word re-evaluation of every primary hit
    other_flags = base_flags if args.accurate else base_flags | V.RENDER_ACCURATE_NORMALS
    for _ in range(args.warmup):
        ctx.render(tlas, cam, W, H, image.data_ptr(), flags=other_flags, stream=sp)
    torch.cuda.synchronize()
    e0.record(stream)
    for _ in range(args.steps):
        ctx.render(tlas, cam, W, H, image.data_ptr(), flags=other_flags, stream=sp)
    e1.record(stream)
    torch.cuda.synchronize()
    ms_other = e0.elapsed_time(e1) / args.steps
    other = {"ms_per_step": round(ms_other, 4), "value": round(rays / (ms_other * 1e-3) / 1e6, 3), "unit": "Mrays/s",
             "frame_time_vs_headline": round(ms_other / ms, 3),
             "normals": "FP32 (miss the 1e-4 rad bound against FP64)" if args.accurate
             else "double-word re-evaluation (within 1e-4 rad of FP64)"}
    log(f"[bench] {'FP32-only' if args.accurate else 'accurate'} frame: {ms_other:.3f} ms, {other['value']:.1f} Mrays/s")

    roofline = None
    if not args.no_roofline:
        roofline = roofline_block(ctx, tlas, cam, W, H, args.polish, kavg, sp, torch, np, V, args.accurate)

    collapse = None
    if not args.no_collapse_study:
        collapse = collapse_block(args, ctx, cam, W, H, flags, sp, stream, torch, np, V, curves, nseg_total)
        ctx.set_option(V.OPTION_BVH_COLLAPSE, tuning["bvh_collapse"] if tuning else 0)

    # the autotuned BVH settings belong to the 100k-strand scene; the other workloads build
    # their BVHs with the library defaults (8 children, leaf size 1, greedy collapse)
    ctx.set_option(V.OPTION_BVH_WIDTH, 8)
    ctx.set_option(V.OPTION_LEAF_SIZE, 1)
    ctx.set_option(V.OPTION_BVH_COLLAPSE, 0)

    modes = None
    if not args.no_modes:
        modes = geometry_modes_block(args, ctx, tlas, cam, W, H, ms, sp, stream, torch, V, curves, nseg_total)

    neural = None
    if not args.no_neural:
        neural = neural_block(args, ctx, tlas, cam, W, H, flags, ms, sp, stream, torch, np, V, curves, nseg_total)

    batch = None
    if not args.no_batch:
        batch = batch_block(args, ctx, sp, stream, torch, V)

    area = None
    if not args.no_area:
        area = neural_area_block(args, ctx, sp, stream, torch, np, V)

    cpu = None
    parity = None
    if not args.no_cpu_baseline:
        cpu, parity = cpu_baseline(args, ctx, tlas, cam, W, H, flags, sp, torch, np, V, curves)

    out = {
        "metric": METRIC,
        "value": round(mrays, 3),
        "unit": "Mrays/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic (seeded strand generator, per-strand SplitMix64)",
        "config": {
            "workload": "phantom_100k_strands_x32_segments_1920x1080_primary_plus_shadow",
            "strands": NS, "segments_per_strand": SEG, "segments": nseg_total,
            "width": W, "height": H, "geometry": "phantom_cubic_bezier",
            "radius": "per-point taper 0.04->0.01", "fp64_polish": bool(args.polish),
            "accurate_normals": bool(args.accurate),
            "rays_per_frame": rays, "primary_rays": n_primary, "shadow_rays": n_shadow,
            "bvh": {"width": tuning["bvh_width"] if tuning else 8,
                    "collapse": ("greedy" if tuning["bvh_collapse"] == 0 else
                                 f"sah_prim_cost_{tuning['bvh_collapse'] / 4:g}") if tuning else "greedy",
                    "leaf_size": tuning["leaf_size"] if tuning else args.leaf_size, "nodes": binfo["node_count"],
                    "depth": binfo["depth"], "build_ms": round(binfo["build_ms"], 3)},
            "stack_kind": tuning["stack_kind"] if tuning else args.stack_kind, "persistent": bool(args.persistent),
            "refill_min": tuning["refill_min"] if tuning else args.refill_min,
            "blocks_per_cu": tuning["blocks_per_cu"] if tuning else args.blocks_per_cu,
            "ray_order": tuning["ray_order"] if tuning else args.ray_order,
            "xcd_chunk": tuning["xcd_chunk"] if tuning else args.xcd_chunk,
            "steps_per_iteration": tuning["steps_per_iteration"] if tuning else args.steps_per_iteration,
            "autotune": tuning,
        },
        "roofline": roofline,
        ("fp32_normals" if args.accurate else "accurate_normals"): other,
        "cpu_baseline": cpu,
        "neural": neural,
        "geometry_modes": modes,
        "bvh_collapse": collapse,
        "batch": batch,
        "neural_area_light": area,
    }
    if parity is not None:
        out["parity_sample"] = parity
    if roofline is not None and roofline.get("work") and parity is not None and parity.get("flop_census"):
        roofline["valu"] = valu_block(roofline, parity["flop_census"])
    print(json.dumps(out), flush=True)
    ctx.close()


def neural_block(args, ctx, tlas, cam, W, H, flags, exact_ms, sp, stream, torch, np, V, curves, nseg):
    """Neural shadow form: the MLP trained on shadow rays the exact tracer labels from
    `neural_views` cameras around the hair (the bench camera is not among them), then frames
    rendered with the variance-gated MLP. The threshold is the largest of a fixed list whose
    frame sends part of the queries to the exact fallback and stays at PSNR >= 40 dB against
    the exact image of the same frame."""
    cv = curves.view(-1, 4, 4)[:, :, :3].reshape(-1, 3)
    lo = cv.min(0).values.tolist()
    hi = cv.max(0).values.tolist()
    pad = [0.05 * (b - a) + 1.0 for a, b in zip(lo, hi)]
    mlp = V.ShadowMLP(ctx, [a - p for a, p in zip(lo, pad)], [b + p for b, p in zip(hi, pad)], seed=1)
    TW, TH = 960, 540
    n = TW * TH
    rays = torch.empty(n * 8, dtype=torch.float32, device="cuda")
    hits = torch.empty(n * 8, dtype=torch.float32, device="cuda")
    srays = torch.empty(n * 8, dtype=torch.float32, device="cuda")
    cnt = torch.zeros(1, dtype=torch.int32, device="cuda")
    samples, targets = [], []
    t0 = time.perf_counter()
    for k in range(args.neural_views):
        a = 2 * math.pi * (k + 0.5) / args.neural_views
        eye = (320 * math.sin(a), 40.0 + 120 * math.sin(3 * a + 0.7), 320 * math.cos(a))
        vc = V.camera_look_at(eye, (0.0, 40.0, 0.0), fov_deg=60.0, aspect=TW / TH)
        ctx.generate_camera_rays(vc, TW, TH, rays.data_ptr(), stream=sp)
        ctx.trace_rays(tlas, rays.data_ptr(), n, hits.data_ptr(), 0, sp)
        cnt.zero_()
        ctx.generate_shadow_rays(rays.data_ptr(), hits.data_ptr(), n, srays.data_ptr(), cnt.data_ptr(), stream=sp)
        torch.cuda.synchronize()
        m = int(cnt.item())
        smp = torch.empty(m * 8, dtype=torch.float32, device="cuda")
        tgt = torch.empty(m, dtype=torch.float32, device="cuda")
        mlp.collect(tlas, srays.data_ptr(), m, smp.data_ptr(), tgt.data_ptr(), stream=sp)
        samples.append(smp)
        targets.append(tgt)
    smp = torch.cat(samples).contiguous()
    tgt = torch.cat(targets).contiguous()
    torch.cuda.synchronize()
    collect_s = time.perf_counter() - t0
    ns = tgt.numel()
    del rays, hits, srays, samples, targets
    t0 = time.perf_counter()
    loss = mlp.train(smp.data_ptr(), tgt.data_ptr(), ns, batch=65536, epochs=args.neural_epochs,
                     learning_rate=3e-3, stream=sp)
    train_s = time.perf_counter() - t0
    train_tflops = 3 * 36992 * ns * args.neural_epochs / train_s / 1e12  # forward + backward ~ 3x forward
    log(f"[bench] neural: {ns} shadow samples from {args.neural_views} views ({collect_s:.2f} s), "
        f"{args.neural_epochs} epochs in {train_s:.2f} s, loss {loss:.4f}")

    # exact and neural float images of the bench frame for PSNR
    fimg_exact = torch.zeros(W * H * 4, dtype=torch.float32, device="cuda")
    ctx.render(tlas, cam, W, H, fimg_exact.data_ptr(), flags=flags & ~V.RENDER_RGBA8, stream=sp)
    torch.cuda.synchronize()
    exact_img = fimg_exact.view(H, W, 4)[..., :3]
    fimg = torch.zeros(W * H * 4, dtype=torch.float32, device="cuda")

    def psnr_at(thr):
        ctx.render(tlas, cam, W, H, fimg.data_ptr(), flags=(flags & ~V.RENDER_RGBA8) | V.RENDER_NEURAL_SHADOWS,
                   shadow_mlp=mlp, variance_threshold=thr, stream=sp)
        torch.cuda.synchronize()
        mse = float(((fimg.view(H, W, 4)[..., :3] - exact_img) ** 2).mean())
        _, q, tr = ctx.render_stats()
        return (float("inf") if mse == 0 else 10 * math.log10(1.0 / mse)), q, tr

    sweep = []
    chosen = None
    for thr in NEURAL_THRESHOLDS:
        p, q, tr = psnr_at(thr)
        sweep.append({"threshold": thr, "psnr_db": round(p, 2) if math.isfinite(p) else None,
                      "fallback_fraction": round(tr / max(q, 1), 4)})
        if p >= 40.0 and tr > 0 and chosen is None:
            chosen = (thr, p, q, tr)
    thr, p, q, tr = chosen if chosen else (0.0,) + psnr_at(0.0)
    image = torch.empty(W * H, dtype=torch.int32, device="cuda")
    nflags = flags | V.RENDER_NEURAL_SHADOWS

    def frame():
        ctx.render(tlas, cam, W, H, image.data_ptr(), flags=nflags, shadow_mlp=mlp, variance_threshold=thr, stream=sp)

    for _ in range(args.warmup):
        frame()
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record(stream)
    for _ in range(args.steps):
        frame()
    e1.record(stream)
    torch.cuda.synchronize()
    ms = e0.elapsed_time(e1) / args.steps
    prim, queries, traced = ctx.render_stats()
    ctx.profiling(True)
    for _ in range(args.steps):
        frame()
    torch.cuda.synchronize()
    shadow_stage = ctx.kernel_stats("render_shadow")
    ctx.profiling(False)
    stage_ms = shadow_stage[0] / max(shadow_stage[1], 1)
    log(f"[bench] neural: threshold {thr} PSNR {p:.2f} dB, fallback {traced}/{queries}, {ms:.3f} ms/frame "
        f"(exact {exact_ms:.3f}), shadow stage {stage_ms:.3f} ms")
    mlp.close()
    return {
        "ms_per_step": round(ms, 4),
        "value": round((prim + queries) / (ms * 1e-3) / 1e6, 3),
        "unit": "Mrays/s (primary rays + shadow queries)",
        "frame_speedup_vs_exact": round(exact_ms / ms, 3),
        "psnr_db_vs_exact": round(p, 2) if math.isfinite(p) else None,
        "variance_threshold": thr,
        "shadow_queries": queries,
        "shadow_rays_traced": traced,
        "shadow_stage_ms": round(stage_ms, 4),
        "threshold_sweep": sweep,
        "train": {"samples": ns, "views": args.neural_views, "epochs": args.neural_epochs, "batch": 65536,
                  "seconds": round(train_s, 3), "collect_seconds": round(collect_s, 3),
                  "final_loss": round(loss, 5), "approx_tflops": round(train_tflops, 2)},
        "held_out": "bench camera is not among the training views",
    }


def geometry_modes_block(args, ctx, tlas, cam, W, H, phantom_ms, sp, stream, torch, V, curves, nseg):
    """The same hair and frame in the other geometry modes: every cubic segment split into
    4 linear pieces (12.8M at 3.2M segments), traced as Linear Swept Spheres (one capsule per
    piece), as DOTS (2 orthogonal quads = 4 triangles per piece) and as voxels (the pieces
    voxelized as capsules of radius 0.02 into cells of --voxel-size, walked by the DDA).
    Reported per mode: build time, frame time and Mrays/s of the exact primary + shadow frame,
    and the PSNR of its float image against the phantom image of the same frame (the image
    error the mode trades)."""
    pieces = nseg * 4
    pl = torch.empty(pieces * 8, dtype=torch.float32, device="cuda")
    ctx.curves_to_lines(curves.data_ptr(), nseg, 4, pl.data_ptr(), stream=sp)
    fimg = torch.zeros(W * H * 4, dtype=torch.float32, device="cuda")
    ctx.render(tlas, cam, W, H, fimg.data_ptr(), flags=V.RENDER_SHADOWS | V.RENDER_FP64_POLISH, stream=sp)
    torch.cuda.synchronize()
    phantom_img = fimg.view(H, W, 4)[..., :3].clone()
    image = torch.empty(W * H, dtype=torch.int32, device="cuda")
    out = {}
    for mode, name in ((V.GEOMETRY_LSS, "lss"), (V.GEOMETRY_DOTS, "dots"), (V.GEOMETRY_VOXELS, "voxels")):
        if mode == V.GEOMETRY_LSS:
            prims = torch.empty(pieces * 8, dtype=torch.float32, device="cuda")
            ctx.generate_lss(pl.data_ptr(), pieces, prims.data_ptr(), stream=sp)
        else:
            prims = pl  # the DOTS and voxel BLASes take the lines and build on the device
        blas = V.BottomLevelAccelerationStructure(ctx, mode, prims.data_ptr(), pieces, leaf_size=args.leaf_size,
                                                  voxel_size=args.voxel_size, stream=sp)
        mtlas = V.TopLevelAccelerationStructure(ctx, [blas], stream=sp)
        torch.cuda.synchronize()
        info = blas.info()

        def frame():
            ctx.render(mtlas, cam, W, H, image.data_ptr(), flags=V.RENDER_SHADOWS | V.RENDER_RGBA8, stream=sp)

        for _ in range(args.warmup):
            frame()
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record(stream)
        for _ in range(args.steps):
            frame()
        e1.record(stream)
        torch.cuda.synchronize()
        ms = e0.elapsed_time(e1) / args.steps
        ctx.synchronize(sp)  # raises on traversal stack overflow
        n_primary, n_shadow = ctx.render_ray_counts()
        fimg.zero_()
        ctx.render(mtlas, cam, W, H, fimg.data_ptr(), flags=V.RENDER_SHADOWS, stream=sp)
        torch.cuda.synchronize()
        mse = float(((fimg.view(H, W, 4)[..., :3] - phantom_img) ** 2).mean())
        psnr = float("inf") if mse == 0 else 10 * math.log10(1.0 / mse)
        mrays = (n_primary + n_shadow) / (ms * 1e-3) / 1e6
        log(f"[bench] {name}: {pieces} pieces, build {info['build_ms']:.1f} ms, depth {info['depth']}, "
            f"{ms:.3f} ms/frame, {mrays:.1f} Mrays/s, PSNR vs phantom {psnr:.2f} dB")
        if mode == V.GEOMETRY_VOXELS:
            cells, _, cell = blas.voxel_grid()
            voxel_info = {"voxel_size": cell, "grid": list(cells.shape[::-1]), "filled": int(info["leaf_records"])}
            log(f"[bench] voxels: grid {voxel_info['grid']} of {cell} cells, {voxel_info['filled']} filled")
        out[name] = {
            "pieces": pieces,
            "triangles": pieces * 4 if mode == V.GEOMETRY_DOTS else None,
            "ms_per_step": round(ms, 4),
            "value": round(mrays, 3),
            "unit": "Mrays/s",
            "frame_time_vs_phantom": round(ms / phantom_ms, 3),
            "primary_rays": n_primary, "shadow_rays": n_shadow,
            "psnr_db_vs_phantom": round(psnr, 2) if math.isfinite(psnr) else None,
            "bvh": {"nodes": info["node_count"], "depth": info["depth"], "build_ms": round(info["build_ms"], 3),
                    "device_bytes": info["device_bytes"]},
        }
        if mode == V.GEOMETRY_VOXELS:
            out[name]["triangles"] = None
            out[name]["voxels"] = voxel_info
        mtlas.close()
        blas.close()
        del prims
    return out


def collapse_block(args, ctx, cam, W, H, flags, sp, stream, torch, np, V, curves, nseg):
    """The binary tree collapsed to 8-wide nodes by the greedy rule (open the largest-area
    child) and by the SAH-optimal rule at primitive costs 0.25, 0.5 and 1 (node cost 1): wide
    nodes, build time, nodes visited and records tested per primary ray of the frame (one
    thread per ray, closest hit), and the frame time (the headline frame's flags) of the phantom
    hair and of its LSS and DOTS forms (12.8M pieces)."""
    n = W * H
    rays = torch.empty(n * 8, dtype=torch.float32, device="cuda")
    hits = torch.empty(n * 8, dtype=torch.float32, device="cuda")
    stats = torch.empty(n * 2, dtype=torch.int32, device="cuda")
    image = torch.empty(n, dtype=torch.int32, device="cuda")
    ctx.generate_camera_rays(cam, W, H, rays.data_ptr(), stream=sp)
    pieces = nseg * 4
    pl = torch.empty(pieces * 8, dtype=torch.float32, device="cuda")
    ctx.curves_to_lines(curves.data_ptr(), nseg, 4, pl.data_ptr(), stream=sp)
    caps = torch.empty(pieces * 8, dtype=torch.float32, device="cuda")
    ctx.generate_lss(pl.data_ptr(), pieces, caps.data_ptr(), stream=sp)
    forms = [("phantom", V.GEOMETRY_PHANTOM_CURVES, curves, nseg, V.BLAS_PER_POINT_RADIUS, flags),
             ("lss", V.GEOMETRY_LSS, caps, pieces, 0, V.RENDER_SHADOWS | V.RENDER_RGBA8),
             ("dots", V.GEOMETRY_DOTS, pl, pieces, V.BLAS_PER_POINT_RADIUS, V.RENDER_SHADOWS | V.RENDER_RGBA8)]
    out = {}
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    for name, mode, prims, count, bflags, rflags in forms:
        rows = {}
        for coll in (0, 1, 2, 4):
            ctx.set_option(V.OPTION_BVH_COLLAPSE, coll)
            blas = V.BottomLevelAccelerationStructure(ctx, mode, prims.data_ptr(), count, flags=bflags, stream=sp)
            tlas = V.TopLevelAccelerationStructure(ctx, [blas], stream=sp)
            torch.cuda.synchronize()
            info = blas.info()
            ctx.trace_stats(tlas, rays.data_ptr(), n, hits.data_ptr(), stats.data_ptr(), stream=sp)
            torch.cuda.synchronize()
            st = stats.view(n, 2).to(torch.float64).mean(0).tolist()
            for _ in range(args.warmup):
                ctx.render(tlas, cam, W, H, image.data_ptr(), flags=rflags, stream=sp)
            e0.record(stream)
            for _ in range(args.steps):
                ctx.render(tlas, cam, W, H, image.data_ptr(), flags=rflags, stream=sp)
            e1.record(stream)
            torch.cuda.synchronize()
            ms = e0.elapsed_time(e1) / args.steps
            key = "greedy" if coll == 0 else f"sah_prim_cost_{coll / 4:g}"
            rows[key] = {"nodes": info["node_count"], "depth": info["depth"], "build_ms": round(info["build_ms"], 3),
                         "nodes_visited_per_ray": round(st[0], 3), "records_tested_per_ray": round(st[1], 3),
                         "ms_per_frame": round(ms, 4)}
            log(f"[bench] collapse {name} {key}: {rows[key]}")
            tlas.close()
            blas.close()
        out[name] = rows
    return out


def copy_calibration(nbytes):
    """A unit-scale elementwise copy (reads nbytes, writes nbytes per launch), 4x larger than the
    256 MB last-level cache so both sides go to HBM."""
    import torch
    n = nbytes // 4
    src = torch.ones(n, dtype=torch.float32, device="cuda")
    dst = torch.empty_like(src)
    torch.cuda.synchronize()
    for _ in range(3):
        torch.mul(src, 1.0, out=dst)
    torch.cuda.synchronize()
    print(json.dumps({"copy_calibration_bytes_read": n * 4, "bytes_written": n * 4, "launches": 3}), flush=True)


def work_counts(args_frames=3, accurate=1):
    """Work counters of the same frame from the counting build (vkhrt_amd/workcount.py in a
    child process, so its library stays out of this one): per traversal kind the node tests,
    leaf early-out tests, Prhi calls, lane use and the split of wave clock cycles."""
    import subprocess
    r = subprocess.run([sys.executable, "-m", "vkhrt_amd.workcount", "--frames", str(args_frames),
                        "--accurate", str(int(accurate))], cwd=ROOT, capture_output=True, text=True, timeout=300)
    if r.returncode != 0:
        log(f"[bench] work counters unavailable: {r.stderr.strip()[-300:]}")
        return None
    return json.loads(r.stdout.strip().splitlines()[-1])


def valu_block(roofline, census):
    """Useful FP32 work of the dominant kernel against the FP32 peak: the GPU's counts of node
    tests, leaf early-out tests, Prhi calls and rays (counting build, same frame) times the FLOP
    each takes (node test: NODE_TEST_FLOP from the kernel's arithmetic; ray frame, early-out and
    Prhi: the oracle's templates run with an operation-counting float on sampled rays of the
    frame, Prhi averaged over its calls), divided by the kernel's average time."""
    w = roofline["work"]["primary"]["per_frame"]
    fl = {"node_test": NODE_TEST_FLOP,
          "ray_frame": census["frame_flop"] / census["rays"],
          "early_out": census["early_out_flop"] / max(census["early_out_tests"], 1),
          "prhi_call": census["prhi_flop"] / max(census["prhi_calls"], 1)}
    parts = {"node_tests": w["node_tests"] * fl["node_test"], "early_out": w["leaf_tests"] * fl["early_out"],
             "prhi": w["prhi_calls"] * fl["prhi_call"], "ray_frames": w["rays"] * fl["ray_frame"]}
    total = sum(parts.values())
    ms = roofline["kernel_avg_ms"]["render_primary"]
    achieved = total / (ms * 1e-3) / 1e12
    return {"bound": "valu", "kernel": "render_primary", "achieved": round(achieved, 3), "peak": FP32_PEAK_TFLOPS,
            "unit": "TFLOP/s", "frac": round(achieved / FP32_PEAK_TFLOPS, 5),
            "useful_flop_per_launch": round(total), "flop_each": {k: round(v, 1) for k, v in fl.items()},
            "share": {k: round(v / total, 4) for k, v in parts.items()},
            "prhi_iterations_per_call": round(census["prhi_iterations"] / max(census["prhi_calls"], 1), 2),
            "lane_use": roofline["work"]["primary"]["lane_use"],
            "wave_cycle_share": roofline["work"]["primary"]["cycle_share"],
            "note": "useful = the arithmetic the method needs; the kernel also spends VALU slots on idle lanes, "
                    "integer decoding, queues and control (see wave_cycle_share, lane_use)"}


def roofline_block(ctx, tlas, cam, W, H, polish, kavg, sp, torch, np, V, accurate=1):
    """Algorithmic bytes per launch of the dominant kernel / its average duration."""
    n = W * H
    rays = torch.empty(n * 8, dtype=torch.float32, device="cuda")
    hits = torch.empty(n * 8, dtype=torch.float32, device="cuda")
    counts = torch.empty(n, dtype=torch.int32, device="cuda")
    ctx.generate_camera_rays(cam, W, H, rays.data_ptr(), stream=sp)
    tflags = V.TRACE_FP64_POLISH if polish else 0
    ctx.trace_rays(tlas, rays.data_ptr(), n, hits.data_ptr(), tflags, sp)
    ctx.count_candidates(tlas, rays.data_ptr(), hits.data_ptr(), n, counts.data_ptr(), stream=sp)
    torch.cuda.synchronize()
    nstar_primary = counts.to(torch.int64).sum().item()
    # shadow rays of the frame, counted against their closest hit
    srays = torch.empty(n * 8, dtype=torch.float32, device="cuda")
    scount = torch.zeros(1, dtype=torch.int32, device="cuda")
    ctx.generate_shadow_rays(rays.data_ptr(), hits.data_ptr(), n, srays.data_ptr(), scount.data_ptr(),
                             stream=sp)
    torch.cuda.synchronize()
    ns = int(scount.item())
    shits = torch.empty(max(1, ns) * 8, dtype=torch.float32, device="cuda")
    ctx.trace_rays(tlas, srays.data_ptr(), ns, shits.data_ptr(), tflags, sp)
    ctx.count_candidates(tlas, srays.data_ptr(), shits.data_ptr(), ns, counts.data_ptr(), stream=sp)
    torch.cuda.synchronize()
    nstar_shadow = counts[:ns].to(torch.int64).sum().item() if ns else 0
    b_primary = 48 * n + 64 * nstar_primary
    b_shadow = 48 * ns + 64 * nstar_shadow
    prim_ms, shad_ms = kavg["render_primary"], kavg["render_shadow"]
    dom = "render_primary" if prim_ms >= shad_ms else "render_shadow"
    bytes_dom = b_primary if dom == "render_primary" else b_shadow
    ms_dom = max(prim_ms, shad_ms)
    achieved = bytes_dom / (ms_dom * 1e-3) / 1e9 if ms_dom > 0 else 0.0
    log(f"[bench] N*_prim primary {nstar_primary / n:.3f}/ray, shadow {nstar_shadow / max(1, ns):.3f}/ray; "
        f"dominant {dom}: {bytes_dom / 1e6:.1f} MB in {ms_dom:.3f} ms -> {achieved:.1f} GB/s")
    work = work_counts(args_frames=3, accurate=accurate)
    traffic = None
    tpath = os.path.join(ROOT, "profiles", "render_primary_phantom_c1_traffic.json")
    if os.path.exists(tpath):
        with open(tpath) as f:
            t = json.load(f)
        traffic = t.get(dom + "_hbm_bytes")
    return {
        "bound": "hbm",
        "kernel": dom,
        "achieved": round(achieved, 2),
        "peak": HBM_PEAK_GBS,
        "unit": "GB/s",
        "frac": round(achieved / HBM_PEAK_GBS, 5),
        "traffic": traffic,
        "traffic_source": "HBM bytes per launch counted in an earlier run of these kernels "
                          "(profiles/render_primary_phantom_c1_traffic.md), not in this one" if traffic else None,
        "basis": "per ray 32 B ray + 16 B hit + 64 B x N*_prim (segments whose exact AABB "
                 "overlaps [tmin, t_closest])",
        "algorithmic_bytes": {"render_primary": b_primary, "render_shadow": b_shadow},
        "nstar_per_ray": {"primary": round(nstar_primary / n, 4),
                          "shadow": round(nstar_shadow / max(1, ns), 4)},
        "kernel_avg_ms": {k: round(v, 4) for k, v in kavg.items()},
        "work": work,
    }


BATCH_MODELS = [(10000, 101), (50000, 102), (200000, 103), (500000, 104)]  # (strands, seed), 32 segments
BATCH_RES = [(512, 512), (1024, 576), (1280, 720), (1920, 1080)]
BATCH_TINTS = [(1.0, 1.0, 1.0), (0.9, 0.7, 0.5), (0.6, 0.8, 1.0), (1.0, 0.6, 0.6)]


def batch_block(args, ctx, sp, stream, torch, V):
    """Batched form: 4 seeded hair models of uneven size (10k / 50k / 200k / 500k strands x 32
    segments = 24.32M segments) side by side as instances of one TLAS (material = model), and 64
    views (16 orbiting each model) at mixed resolutions 512x512 .. 1920x1080 = 61.5M paths,
    path traced with 4 bounces through one pipeline (global path queue, one persistent traversal
    launch per depth for all views) captured as a HIP graph. value = traced rays (primary +
    bounce + shadow) per second."""
    nseg = 32
    blases, keep = [], []
    t0 = time.perf_counter()
    for k, (ns, seed) in enumerate(BATCH_MODELS):
        n = ns * nseg
        verts = torch.empty(ns * (nseg + 1) * 4, dtype=torch.float32, device="cuda")
        lines = torch.empty(n * 8, dtype=torch.float32, device="cuda")
        curves = torch.empty(n * 16, dtype=torch.float32, device="cuda")
        ctx.generate_strands(seed, ns, nseg, verts.data_ptr(), stream=sp)
        ctx.generate_lines(verts.data_ptr(), ns, nseg, lines.data_ptr(), stream=sp)
        ctx.generate_curves(lines.data_ptr(), n, curves.data_ptr(), stream=sp)
        xf = [1.0, 0.0, 0.0, 500.0 * k - 750.0, 0.0, 1.0, 0.0, 0.0, 0.0, 0.0, 1.0, 0.0]
        blases.append(V.BottomLevelAccelerationStructure(ctx, V.GEOMETRY_PHANTOM_CURVES, curves.data_ptr(), n,
                                                         flags=V.BLAS_PER_POINT_RADIUS, transform=xf,
                                                         material_index=k, leaf_size=args.leaf_size, stream=sp))
        del verts, lines, curves
    tlas = V.TopLevelAccelerationStructure(ctx, blases, stream=sp)
    torch.cuda.synchronize()
    build_s = time.perf_counter() - t0
    views, images = [], []
    for v in range(64):
        k, j = v % 4, v // 4
        w, h = BATCH_RES[(v + j) % 4]
        a = 2 * math.pi * (j + 0.5) / 16
        cx = 500.0 * k - 750.0
        eye = (cx + 280 * math.sin(a), 60.0 + 90 * math.sin(3 * a), 280 * math.cos(a))
        cam = V.camera_look_at(eye, (cx, 40.0, 0.0), fov_deg=60.0, aspect=w / h)
        img = torch.empty(w * h, dtype=torch.int32, device="cuda")
        images.append(img)
        views.append((cam, w, h, img.data_ptr()))
    paths = sum(w * h for _, w, h, _ in views)
    base = V.BATCH_RGBA8 | V.BATCH_FP64_POLISH

    def timed(flags, frames, seed0=0):
        for i in range(max(1, args.warmup // 2)):
            ctx.render_batch(tlas, views, bounces=4, seed=seed0 + i, environment=(0.25, 0.3, 0.35), flags=flags,
                             material_albedo=BATCH_TINTS, stream=sp)
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record(stream)
        for i in range(frames):
            ctx.render_batch(tlas, views, bounces=4, seed=seed0 + 100 + i, environment=(0.25, 0.3, 0.35),
                             flags=flags, material_albedo=BATCH_TINTS, stream=sp)
        e1.record(stream)
        torch.cuda.synchronize()
        ctx.synchronize(sp)
        _, nb, nshadow, caps = ctx.batch_stats()
        return e0.elapsed_time(e1) / frames, nb, nshadow, caps

    frames = max(2, min(args.steps, 5))
    tuned = None
    if args.autotune:
        t0 = time.perf_counter()
        tuned = ctx.autotune_batch(tlas, views, bounces=4, seed=0, environment=(0.25, 0.3, 0.35),
                                   flags=base | V.BATCH_GRAPH, material_albedo=BATCH_TINTS, repeats=1, stream=sp)
        tuned["seconds"] = round(time.perf_counter() - t0, 2)
        log(f"[bench] batch autotuned: {tuned}")
    variants = {}
    named = [("autotuned", base | V.BATCH_GRAPH | tuned["batch_flags"])] if tuned else []
    for name, fl in named + [("graph_raysort", base | V.BATCH_GRAPH | V.BATCH_SORT_RAYS),
                     ("graph_raysort_material", base | V.BATCH_GRAPH | V.BATCH_SORT_RAYS | V.BATCH_SORT_MATERIALS),
                     ("graph", base | V.BATCH_GRAPH), ("eager", base)]:
        ms, nb, nshadow, caps = timed(fl, frames)
        rays = paths + nb + nshadow
        variants[name] = {"ms_per_frame": round(ms, 3), "mrays_per_s": round(rays / (ms * 1e-3) / 1e6, 1),
                          "bounce_rays": nb, "shadow_rays": nshadow}
        log(f"[bench] batch {name}: {ms:.2f} ms/frame, {paths} paths + {nb} bounce + {nshadow} shadow rays "
            f"-> {rays / (ms * 1e-3) / 1e6:.1f} Mrays/s (graph captures {caps})")
    best = min(variants, key=lambda k: variants[k]["ms_per_frame"])
    tlas.close()
    for b in blases:
        b.close()
    return {
        "workload": "4_models_10k_50k_200k_500k_strands_x32_64_views_512_to_1080p_4_bounces",
        "segments": sum(ns for ns, _ in BATCH_MODELS) * nseg, "views": 64, "paths": paths, "bounces": 4,
        "build_seconds": round(build_s, 3),
        "value": variants[best]["mrays_per_s"], "unit": "Mrays/s (primary + bounce + shadow rays)",
        "ms_per_frame": variants[best]["ms_per_frame"], "best": best, "variants": variants,
        "fp64_polish": True, "autotune": tuned,
    }


AREA_LIGHT = ((0.0, 260.0, 0.0), (100.0, 0.0, 0.0), (0.0, 0.0, 100.0))  # center, edge u, edge v
# variance thresholds of the neural sweeps, largest first (p (1 - p) never exceeds 0.25)
NEURAL_THRESHOLDS = (0.2499, 0.249, 0.245, 0.24, 0.23, 0.22, 0.2, 0.15, 0.1, 0.05, 0.02, 0.0)


def neural_area_block(args, ctx, sp, stream, torch, np, V):
    """Neural shadow form on the 500k-strand x 32-segment model (16M segments) at 1920x1080
    with 2 area-light samples per hit. The MLP is trained (Adam, BF16 MFMA forward/backward) on
    2^24 shadow rays from points drawn uniformly on the strand surfaces toward light points,
    labelled by the exact tracer; evaluated on 2^20 held-out rays (another seed); then the frame
    is rendered with the variance-gated MLP (exact fallback above the threshold) against the
    exact frame."""
    ns, nseg, seed = 500000, 32, 104
    n = ns * nseg
    verts = torch.empty(ns * (nseg + 1) * 4, dtype=torch.float32, device="cuda")
    lines = torch.empty(n * 8, dtype=torch.float32, device="cuda")
    curves = torch.empty(n * 16, dtype=torch.float32, device="cuda")
    ctx.generate_strands(seed, ns, nseg, verts.data_ptr(), stream=sp)
    ctx.generate_lines(verts.data_ptr(), ns, nseg, lines.data_ptr(), stream=sp)
    ctx.generate_curves(lines.data_ptr(), n, curves.data_ptr(), stream=sp)
    del verts, lines
    blas = V.BottomLevelAccelerationStructure(ctx, V.GEOMETRY_PHANTOM_CURVES, curves.data_ptr(), n,
                                              flags=V.BLAS_PER_POINT_RADIUS, stream=sp)
    tlas = V.TopLevelAccelerationStructure(ctx, [blas], stream=sp)
    cv = curves.view(-1, 4, 4)[:, :, :3].reshape(-1, 3)
    lo, hi = cv.min(0).values.tolist(), cv.max(0).values.tolist()
    del cv
    torch.cuda.synchronize()
    W, H = args.width, args.height
    cam = V.camera_look_at(CAMERA_EYE, CAMERA_TARGET, fov_deg=60.0, aspect=W / H)
    light = V.area_light(*AREA_LIGHT, samples=2, seed=7)
    flags = V.RENDER_SHADOWS | V.RENDER_RGBA8 | (V.RENDER_FP64_POLISH if args.polish else 0)
    image = torch.empty(W * H, dtype=torch.int32, device="cuda")

    # each form runs with the traversal options the autotuner picked on its own frame
    tunings = {}

    def timed(**kw):
        nflags = flags | (V.RENDER_NEURAL_SHADOWS if kw else 0)
        tuning = tunings.get("neural" if kw else "exact")
        if tuning:
            ctx.apply_tuning(tuning)
        for _ in range(args.warmup):
            ctx.render(tlas, cam, W, H, image.data_ptr(), flags=nflags, stream=sp, area_light=light, **kw)
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record(stream)
        for _ in range(args.steps):
            ctx.render(tlas, cam, W, H, image.data_ptr(), flags=nflags, stream=sp, area_light=light, **kw)
        e1.record(stream)
        torch.cuda.synchronize()
        ctx.synchronize(sp)
        return e0.elapsed_time(e1) / args.steps, ctx.render_stats()

    # the autotuner picks the traversal options on this workload's exact frame, and later on its
    # neural frame; each form is timed with its own
    tune_keys = ("stack_kind", "blocks_per_cu", "refill_min", "ray_order", "xcd_chunk", "steps_per_iteration", "trials")
    area_tuning = neural_tuning = None
    if args.autotune:
        t = ctx.autotune_render(tlas, cam, W, H, image.data_ptr(), flags=flags, repeats=9, stream=sp, area_light=light)
        tunings["exact"] = t
        area_tuning = {k: t[k] for k in tune_keys}
        area_tuning["tuned_ms"] = round(t["best_ms"], 4)
        log(f"[bench] area light autotuned: {area_tuning}")
    exact_ms, (prim, queries, _) = timed()
    log(f"[bench] area light: 16M segments, exact {exact_ms:.3f} ms/frame, {prim} primary + {queries} shadow rays "
        f"-> {(prim + queries) / (exact_ms * 1e-3) / 1e6:.1f} Mrays/s")

    pad = [0.02 * (b - a) + 1.0 for a, b in zip(lo, hi)]
    mlp = V.ShadowMLP(ctx, [a - p for a, p in zip(lo, pad)], [b + p for b, p in zip(hi, pad)], seed=1)
    ntrain, nheld = 1 << 24, 1 << 20

    def data(count, s):
        rays = torch.empty(count * 8, dtype=torch.float32, device="cuda")
        ctx.generate_surface_shadow_rays(tlas, count, s, rays.data_ptr(), light=light, stream=sp)
        smp = torch.empty(count * 8, dtype=torch.float32, device="cuda")
        tgt = torch.empty(count, dtype=torch.float32, device="cuda")
        mlp.collect(tlas, rays.data_ptr(), count, smp.data_ptr(), tgt.data_ptr(), stream=sp)
        torch.cuda.synchronize()
        return smp, tgt

    t0 = time.perf_counter()
    smp, tgt = data(ntrain, 1)
    collect_s = time.perf_counter() - t0
    epochs = 24
    t0 = time.perf_counter()
    loss = mlp.train(smp.data_ptr(), tgt.data_ptr(), ntrain, batch=65536, epochs=epochs, learning_rate=3e-3, stream=sp)
    train_s = time.perf_counter() - t0
    del smp, tgt
    hs, ht = data(nheld, 2)
    p = torch.empty(nheld, dtype=torch.float32, device="cuda")
    mlp.infer(hs.data_ptr(), nheld, p.data_ptr(), stream=sp)
    torch.cuda.synchronize()
    y = ht.double()
    pd = p.double().clamp(1e-7, 1 - 1e-7)
    held = {"rays": nheld, "lit_fraction": round(float(y.mean()), 4),
            "bce": round(float(-(y * pd.log() + (1 - y) * (1 - pd).log()).mean()), 4),
            "accuracy": round(float(((pd > 0.5).double() == y).double().mean()), 4),
            "mean_abs_error": round(float((pd - y).abs().mean()), 4)}
    var = pd * (1 - pd)
    for thr in (0.05, 0.15):
        conf = var <= thr
        held[f"confident_fraction_at_{thr}"] = round(float(conf.double().mean()), 4)
        held[f"error_with_fallback_at_{thr}"] = round(float(((pd - y).abs() * conf).mean()), 4)
    del hs, ht, p
    log(f"[bench] area light: trained on 2^24 surface rays ({collect_s:.2f} s to trace) for {epochs} epochs in "
        f"{train_s:.2f} s, loss {loss:.4f}; held-out {held}")

    if args.autotune:
        t = ctx.autotune_render(tlas, cam, W, H, image.data_ptr(), flags=flags | V.RENDER_NEURAL_SHADOWS, repeats=9,
                                stream=sp, area_light=light, shadow_mlp=mlp, variance_threshold=NEURAL_THRESHOLDS[0])
        tunings["neural"] = t
        neural_tuning = {k: t[k] for k in tune_keys}
        neural_tuning["tuned_ms"] = round(t["best_ms"], 4)
        neural_tuning["threshold"] = NEURAL_THRESHOLDS[0]
        log(f"[bench] area light neural autotuned: {neural_tuning}")
    fimg = torch.zeros(W * H * 4, dtype=torch.float32, device="cuda")
    fexact = torch.zeros(W * H * 4, dtype=torch.float32, device="cuda")
    ctx.render(tlas, cam, W, H, fexact.data_ptr(), flags=flags & ~V.RENDER_RGBA8, stream=sp, area_light=light)
    torch.cuda.synchronize()
    # Every threshold of the sweep is timed, each between two timings of the exact frame: the
    # speed-up compares frames measured in the same few milliseconds (the clock of a long run
    # drifts by a few per cent). p (1 - p) <= 0.25 always, so 0.25 would send no query to the
    # exact fallback; the sweep starts just below it.
    sweep, chosen, exact_all = [], None, [exact_ms]
    for thr in NEURAL_THRESHOLDS:
        ctx.render(tlas, cam, W, H, fimg.data_ptr(), flags=(flags & ~V.RENDER_RGBA8) | V.RENDER_NEURAL_SHADOWS,
                   shadow_mlp=mlp, variance_threshold=thr, stream=sp, area_light=light)
        torch.cuda.synchronize()
        mse = float(((fimg.view(H, W, 4)[..., :3] - fexact.view(H, W, 4)[..., :3]) ** 2).mean())
        psnr = float("inf") if mse == 0 else 10 * math.log10(1.0 / mse)
        e0_ms, _ = timed()
        t_ms, (_, q, tr) = timed(shadow_mlp=mlp, variance_threshold=thr)
        e1_ms, _ = timed()
        e_ms = 0.5 * (e0_ms + e1_ms)
        exact_all += [e0_ms, e1_ms]
        sweep.append({"threshold": thr, "psnr_db": round(psnr, 2) if math.isfinite(psnr) else None,
                      "shadow_rays_traced": tr, "fallback_fraction": round(tr / max(q, 1), 4),
                      "ms_per_step": round(t_ms, 4), "exact_ms_adjacent": round(e_ms, 4),
                      "frame_speedup_vs_exact": round(e_ms / t_ms, 3)})
        log(f"[bench] area light neural: threshold {thr}: PSNR {psnr:.2f} dB, fallback {tr}/{q}, {t_ms:.3f} ms "
            f"(exact {e_ms:.3f}) -> {e_ms / t_ms:.3f}x")
        if chosen is None and psnr >= 40.0 and tr > 0:
            chosen = sweep[-1]
    if chosen is None:
        chosen = sweep[-1]
    thr, psnr, traced, neural_ms = chosen["threshold"], chosen["psnr_db"], chosen["shadow_rays_traced"], \
        chosen["ms_per_step"]
    exact_ms = float(np.median(exact_all))
    q = queries
    log(f"[bench] area light neural: chosen threshold {thr} PSNR {psnr} dB, fallback {traced}/{q}, {neural_ms:.3f} "
        f"ms/frame (exact {chosen['exact_ms_adjacent']:.3f}) -> {chosen['frame_speedup_vs_exact']:.3f}x")
    mlp.close()
    tlas.close()
    blas.close()
    return {
        "workload": "phantom_500k_strands_x32_segments_1920x1080_area_light_2_samples",
        "segments": n, "light_samples": 2, "autotune": area_tuning, "autotune_neural": neural_tuning,
        "exact": {"ms_per_step": round(exact_ms, 4), "primary_rays": prim, "shadow_rays": queries,
                  "mrays_per_s": round((prim + queries) / (exact_ms * 1e-3) / 1e6, 1),
                  "timing": "median of every exact-frame timing of the block"},
        "neural": {"ms_per_step": round(neural_ms, 4), "variance_threshold": thr,
                   "psnr_db_vs_exact": psnr, "shadow_rays_traced": traced, "shadow_queries": q,
                   "exact_ms_adjacent": chosen["exact_ms_adjacent"],
                   "frame_speedup_vs_exact": chosen["frame_speedup_vs_exact"],
                   "choice": "largest threshold of the sweep whose frame traces part of the queries exactly "
                             "and keeps PSNR >= 40 dB against the exact frame",
                   "fallback_walk": {"lanes_per_ray": args.shadow_group_lanes, "queue_limit": 65536},
                   "threshold_sweep": sweep},
        "train": {"samples": ntrain, "epochs": epochs, "batch": 65536, "seconds": round(train_s, 2),
                  "trace_seconds": round(collect_s, 2), "final_loss": round(loss, 5),
                  "approx_tflops": round(3 * 36992 * ntrain * epochs / train_s / 1e12, 2)},
        "held_out": held,
    }


def cpu_baseline(args, ctx, tlas, cam, W, H, flags, sp, torch, np, V, curves_d):
    """The oracle (host C++ transliteration, binned-SAH BVH2) on every k-th pixel of the same
    frame with all host threads; also checks primitive ids against the GPU on that sample."""
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import oracle_lib as O
    L = O.lib()
    threads = L.orc_hardware_threads()
    t0 = time.perf_counter()
    curves = O.hair_curves(args.seed, args.strands, args.segments)
    S = O.Scene()
    S.add(O.MODE_PHANTOM, curves, per_point=True)
    t_build = time.perf_counter() - t0
    vi = np.array(cam.view_inverse, np.float32)
    pi = np.array(cam.proj_inverse, np.float32)
    oflags = (O.F_POLISH if args.polish else 0) | (O.F_ACCURATE if args.accurate else 0)
    # calibrate the sample stride for ~cpu_seconds of tracing
    stride = 997
    _, _, nr, secs = S.render(vi, pi, W, H, flags=oflags, shadows=1, pixel_stride=stride)
    rate = nr / max(secs, 1e-6)
    want = rate * args.cpu_seconds
    per_pix = nr / math.ceil(W * H / stride)
    stride = max(1, int(W * H * per_pix / max(want, 1.0)))
    img, ids, nr, secs = S.render(vi, pi, W, H, flags=oflags, shadows=1, pixel_stride=stride)
    npix = math.ceil(W * H / stride)
    reps = 1
    while secs < args.cpu_seconds and reps < 200:  # whole frame is quick: repeat it
        _, _, nr2, s2 = S.render(vi, pi, W, H, flags=oflags, shadows=1, pixel_stride=stride)
        nr += nr2
        secs += s2
        reps += 1
    value = nr / secs / 1e6
    log(f"[bench] CPU oracle: {npix} pixels (stride {stride}) x{reps}, {nr} rays in {secs:.2f} s on {threads} "
        f"threads -> {value:.3f} Mrays/s (scene+BVH2 {t_build:.1f} s)")
    # GPU primitive ids on the same pixels
    gids = torch.empty(W * H, dtype=torch.int32, device="cuda")
    img_g = torch.empty(W * H, dtype=torch.int32, device="cuda")
    ctx.render(tlas, cam, W, H, img_g.data_ptr(), flags=flags, prim_ids_ptr=gids.data_ptr(), stream=sp)
    torch.cuda.synchronize()
    g = gids.cpu().numpy().view(np.uint32)
    sel = np.arange(0, W * H, stride)
    agree = float((g[sel] == ids.reshape(-1)[sel]).mean())
    hits = int((ids.reshape(-1)[sel] != 0xFFFFFFFF).sum())
    cpu_model = ""
    try:
        with open("/proc/cpuinfo") as f:
            cpu_model = next((ln.split(":", 1)[1].strip() for ln in f if ln.startswith("model name")), "")
    except OSError:
        pass
    cpu = {"value": round(value, 4), "unit": "Mrays/s", "cores": threads, "kind": "port", "cpu_model": cpu_model,
           "sample": f"every {stride}th pixel of the {W}x{H} frame ({npix} pixels) traced {reps} times: "
                     f"{nr} primary+shadow rays in {secs:.1f} s; scene generation + BVH2 build "
                     f"({t_build:.1f} s) excluded"}
    census_rays = O.raygen(vi, pi, W, H)[::97].copy()
    census = S.flop_census(census_rays)
    log(f"[bench] FLOP census on {int(census['rays'])} rays: frame {census['frame_flop'] / census['rays']:.0f}, "
        f"early-out {census['early_out_flop'] / max(census['early_out_tests'], 1):.1f} per test, Prhi "
        f"{census['prhi_flop'] / max(census['prhi_calls'], 1):.0f} per call")
    parity = {"pixels": int(npix), "hit_pixels": hits, "primid_agreement": agree, "flop_census": census,
              "accuracy_vs_fp64": accuracy_sample(ctx, tlas, cam, W, H, args.polish, sp, torch, np, V, O, curves,
                                                  curves_d)}
    return cpu, parity


def accuracy_sample(ctx, tlas, cam, W, H, polish, sp, torch, np, V, O, curves, curves_d, nrays=6000):
    """Hits against the FP64 evaluation of the same intersector (tests/accuracy.py: the oracle's
    Prhi and capsule test in double, the triangle plane in float64), per configuration: the C0
    hair (1,000 strands x 16, its 256x256 view), the C1 frame (FP32 hits and the double-word
    re-run), and the C1 hair as LSS capsules and DOTS quads. Relative t error and normal angle
    (rad) as median / p99 / max."""
    import accuracy as A
    base = V.TRACE_FP64_POLISH if polish else 0

    def trace(tl, rays, fl):
        d_rays = torch.from_numpy(rays.reshape(-1).copy()).cuda()
        h = torch.zeros(rays.shape[0] * 8, dtype=torch.float32, device="cuda")
        ctx.trace_rays(tl, d_rays.data_ptr(), rays.shape[0], h.data_ptr(), fl, sp)
        torch.cuda.synchronize()
        return h.cpu().numpy().view(O.HIT_DTYPE)

    def log_acc(name, a):
        log(f"[bench] vs FP64 ({name}): t rel median {a['t_rel_median']:.2g} p99 {a['t_rel_p99']:.2g} max "
            f"{a['t_rel_max']:.2g}; normal median {a['normal_rad_median']:.2g} p99 {a['normal_rad_p99']:.2g} max "
            f"{a['normal_rad_max']:.2g} rad ({a['hits']} hits)")

    out = {}
    # C0: the 1,000-strand hair and its 256x256 view
    c0 = O.hair_curves(20240601, 1000, 16)
    d0 = torch.from_numpy(c0.reshape(-1).copy()).cuda()
    b0 = V.BottomLevelAccelerationStructure(ctx, V.GEOMETRY_PHANTOM_CURVES, d0.data_ptr(), c0.shape[0],
                                            flags=V.BLAS_PER_POINT_RADIUS, stream=sp)
    t0 = V.TopLevelAccelerationStructure(ctx, [b0], stream=sp)
    vi0, pi0 = O.camera((0.0, 112.0, 140.0), (0.0, 105.0, 0.0), tan_half_fovy=0.2)
    r0 = O.raygen(vi0, pi0, 256, 256)
    for name, fl in (("fp32", base), ("accurate", base | V.TRACE_ACCURATE_NORMALS)):
        out[f"c0_{name}"] = A.phantom(r0, trace(t0, r0, fl), c0, limit=2000)
        log_acc(f"C0 {name}", out[f"c0_{name}"])
    t0.close()
    b0.close()
    # C1: rays spread over the frame
    vi = np.array(cam.view_inverse, np.float32)
    pi = np.array(cam.proj_inverse, np.float32)
    rays = O.raygen(vi, pi, W, H)[np.linspace(0, W * H - 1, nrays * 4).astype(np.int64)]
    for name, fl in (("fp32", base), ("accurate", base | V.TRACE_ACCURATE_NORMALS)):
        out[f"c1_{name}"] = A.phantom(rays, trace(tlas, rays, fl), curves, limit=2000)
        log_acc(f"C1 {name}", out[f"c1_{name}"])
    # C2: the C1 hair as 4 pieces per cubic, LSS capsules and DOTS quads
    n = curves.shape[0] * 4
    pl = torch.empty(n * 8, dtype=torch.float32, device="cuda")
    ctx.curves_to_lines(curves_d.data_ptr(), curves.shape[0], 4, pl.data_ptr(), stream=sp)
    caps = torch.empty(n * 8, dtype=torch.float32, device="cuda")
    ctx.generate_lss(pl.data_ptr(), n, caps.data_ptr(), stream=sp)
    for name, mode, prims, fl in (("c2_lss", V.GEOMETRY_LSS, caps, 0), ("c2_dots", V.GEOMETRY_DOTS, pl,
                                                                        V.BLAS_PER_POINT_RADIUS)):
        b = V.BottomLevelAccelerationStructure(ctx, mode, prims.data_ptr(), n, flags=fl, stream=sp)
        t = V.TopLevelAccelerationStructure(ctx, [b], stream=sp)
        h = trace(t, rays, 0)
        recs = prims.view(n, 8).cpu().numpy()  # 410 MB of records, read back once for the FP64 reference
        out[name] = (A.lss(rays, h, recs, limit=2000) if mode == V.GEOMETRY_LSS
                     else A.dots(rays, h, O.generate_dots(recs), limit=2000))
        del recs
        log_acc(name, out[name])
        t.close()
        b.close()
    return out


if __name__ == "__main__":
    main()
