"""Benchmark: visual hulls/s on one MI355X, batched vs per-scene, with roofline and CPU baseline.

Workload (default, "mixed64"): 64 independent synthetic scenes (1..8 ellipsoids,
4..48 cameras, 256/512/1024 px masks, level 6..9, masks_partial with p=0.3,
blur k=7 sigma=1.5), masks resident in HBM.  One step = sparse blur of every
scene's masks + visual hull of every scene.  `value` is the batched path (one
carving launch per octree level across all scenes); the per-scene path (one
pipeline per scene) is timed on the same data and every batched mesh is
compared with its per-scene mesh.

Prints one JSON line.  Usage: python bench.py [--gpus 1] [--steps K] [--warmup W]
"""

from __future__ import annotations

import argparse
import ctypes
import json
import math
import os
import platform
import statistics
import sys
import threading
import time

import numpy as np
import torch

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

import torchhull_amd as th  # noqa: E402
from torchhull_amd import _lib, synthetic  # noqa: E402

HBM_PEAK_GBS = 8000.0


def log(msg: str) -> None:
    print(msg, file=sys.stderr, flush=True)


def scene_args(sc: synthetic.Scene, masks: torch.Tensor) -> dict:
    return dict(masks=masks, transforms=sc.transforms, level=sc.level, cube_corner_bfl=sc.cube_corner_bfl,
                cube_length=sc.cube_length, masks_partial=sc.masks_partial,
                transforms_convention=sc.transforms_convention)


def blur(sc: synthetic.Scene) -> torch.Tensor:
    if sc.blur is None:
        return sc.masks
    k, s = sc.blur
    return th.gaussian_blur(sc.masks, k, s, sparse=True, dtype=torch.float32)


def step_batched(scenes, graph: bool = True):
    # one blur launch per pass for all scenes (they share k and sigma), then one pipeline for all hulls whose
    # carving loop replays a captured hipGraph (the batch shape repeats every step)
    blurred = th.gaussian_blur_batch([sc.masks for sc in scenes], scenes[0].blur[0], scenes[0].blur[1],
                                     sparse=True, dtype=torch.float32)
    return th.visual_hull_batch([scene_args(sc, m) for sc, m in zip(scenes, blurred)], unique_verts=True,
                                graph=graph)


def step_per_scene(scenes):
    return [th.visual_hull(**scene_args(sc, blur(sc)), unique_verts=True) for sc in scenes]


def timed(fn, steps: int, warmup: int):
    out = None
    for _ in range(warmup):
        out = fn()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        out = fn()
    torch.cuda.synchronize()
    return time.perf_counter() - t0, out


def carve_profile(run_fn, reps: int = 5) -> dict:
    """Runs run_fn `reps` times with event timing of the carving classification launches; per-level
    records with the median time over the runs.  `camera_tests` counts the reference's early-exit tests,
    those of cameras that the solid maps leave out among them: not what a launch reads."""
    ctx = _lib.context(torch.cuda.current_device())
    L = _lib.lib()
    n = 16
    runs = []
    for _ in range(max(1, reps)):
        _lib.check(L.thull_profile_enable(ctx, 1))
        try:
            run_fn()
            torch.cuda.synchronize()
        finally:
            _lib.check(L.thull_profile_enable(ctx, 0))
        ms = (ctypes.c_float * n)()
        par, tests, nxt = (ctypes.c_int64 * n)(), (ctypes.c_int64 * n)(), (ctypes.c_int64 * n)()
        split = (ctypes.c_int32 * n)()
        _lib.check(L.thull_profile_carve(ctx, n, ms, par, tests, nxt, split))
        runs.append((list(ms), list(par), list(tests), list(nxt), list(split)))
    ms_med = [statistics.median(r[0][i] for r in runs) for i in range(n)]
    _, par, tests, nxt, split = runs[-1]
    levels = []
    for i in range(n):
        if par[i] == 0:
            continue
        kernel = {1: "carve_classify_kernel", 0: "carve_classify_queue_kernel", 8: "carve_classify_child_kernel"}.get(
            split[i], f"carve_classify_split_kernel<{split[i]}>")
        levels.append(dict(step=i, level=i + 1, kernel=kernel, ms=float(ms_med[i]), parents=int(par[i]),
                           camera_tests=int(tests[i]), children=int(nxt[i])))
    return dict(levels=levels, reps=len(runs))


CARVE_SOURCES = ("torchhull_amd/csrc/vh_kernels.hip", "torchhull_amd/csrc/common.h", "torchhull_amd/csrc/solid_reach.h",
                 "torchhull_amd/csrc/engine.hip")


def carve_source_hash() -> str:
    """Hash of the sources that decide the carving kernel's memory traffic (kernel, helpers, launch order)."""
    import hashlib

    h = hashlib.sha256()
    for rel in CARVE_SOURCES:
        with open(os.path.join(ROOT, rel), "rb") as f:
            h.update(f.read())
    return h.hexdigest()[:16]


def traffic_from_profile(kernel: str) -> dict | None:
    """HBM bytes per launch of the carving kernel `kernel` in the batched step, from the committed
    rocprofv3 FETCH_SIZE / WRITE_SIZE summary (calibrated against a copy of known size).  The summary
    records the kernel and the hash of the carving sources it was measured on; another kernel or build
    gets {"stale": ...}."""
    path = os.path.join(ROOT, "profiles", "carve_classify_mixed64_traffic.txt")
    try:
        vals = {}
        with open(path) as f:
            for line in f:
                if ":" in line and not line.startswith("#"):
                    k, v = line.split(":", 1)
                    vals[k.strip()] = v.strip()
        if vals.get("carve_source_hash") != carve_source_hash() or vals.get("kernel") != kernel:
            return {"stale": f"{vals.get('kernel')} {vals.get('carve_source_hash')}"}
        return {"fetch": float(vals["fetch_bytes_per_launch"]), "write": float(vals["write_bytes_per_launch"]),
                "hash": vals["carve_source_hash"]}
    except (OSError, KeyError, ValueError):
        return None


def roofline_from(levels: list[dict]) -> dict:
    """Bandwidth of the one-thread-per-parent carving kernel (the largest kernel of the batched step: the
    persistent work-queue kernel of the replayed carving loop) over its launches in one batched step: the
    bytes that its launches move by the hardware counters (traffic_from_profile) over their time here.
    None for a build whose traffic was not measured.  The camera-split launches of the small levels are
    other kernels."""
    name = "carve_classify_queue_kernel" if any(lv["kernel"] == "carve_classify_queue_kernel" for lv in levels) \
        else "carve_classify_kernel"
    sel = [lv for lv in levels if lv["kernel"] == name]
    tot_ms = sum(lv["ms"] for lv in sel)
    n = len(sel)
    tr = traffic_from_profile(name)
    ok = tr is not None and "fetch" in tr
    traffic = int(tr["fetch"] + tr["write"]) if ok else None
    achieved = n * traffic / (tot_ms * 1e-3) / 1e9 if ok and tot_ms > 0 else None
    return {"bound": "hbm", "achieved": None if achieved is None else round(achieved, 1), "peak": HBM_PEAK_GBS,
            "unit": "GB/s", "frac": None if achieved is None else round(achieved / HBM_PEAK_GBS, 4),
            "traffic": traffic,
            "traffic_source": ("profiles/carve_classify_mixed64_traffic.txt, carving sources " + tr["hash"]) if ok
            else ("measured on other carving sources (" + str(tr["stale"]) + "); not reused" if tr else "missing"),
            "kernel": name, "launches": n,
            "levels": [lv["level"] for lv in sel],
            "camera_tests_per_launch": int(sum(lv["camera_tests"] for lv in sel) / max(n, 1)),
            "avg_launch_ms": round(tot_ms / max(n, 1), 4)}


def serve(rate: float, seconds: float, pool_size: int, workers: int, dev: torch.device) -> dict:
    """Open-loop Poisson request stream through the continuous-batching server.

    Requests draw scenes from a pool of mixed-workload scenes with levels 6..10
    (masks resident in HBM); every returned mesh is compared bit for bit with
    the plain per-scene result of its scene."""
    from torchhull_amd import serving

    log(f"serving: rendering a pool of {pool_size} scenes (levels 6..10) ...")
    pool = synthetic.mixed_scenes(pool_size, seed=4000, device=dev, max_level=10)
    plain = [th.visual_hull(**scene_args(sc, blur(sc)), unique_verts=True) for sc in pool]
    torch.cuda.synchronize()
    rng = np.random.default_rng(4001)
    n = int(rate * seconds)
    arrivals = np.cumsum(rng.exponential(1.0 / rate, size=n))
    picks = rng.integers(0, pool_size, size=n)
    lat, batch_sizes, joined = [], [], [0]
    mismatches = [0]
    completed = [0]
    cv = threading.Condition()

    # futures are not kept: each mesh is checked and released as soon as it is done
    def done(fut, k, t_sched):
        ok, r = False, None
        if fut.exception() is None:
            r = fut.result()
            pv, pf = plain[k]
            ok = torch.equal(r.faces, pf) and torch.equal(r.verts.view(torch.int32), pv.view(torch.int32))
        with cv:
            if r is not None:
                lat.append(r.finished - t_sched)
                batch_sizes.append(r.batch_size)
                joined[0] += 1 if r.joined_step > 0 else 0
            if not ok:
                mismatches[0] += 1
            completed[0] += 1
            cv.notify_all()

    log(f"serving: {n} requests at {rate:.0f} req/s for {seconds:.0f} s, {workers} workers ...")
    with serving.HullServer(dev, workers=workers) as srv:
        # warm-up: one request per worker, not counted
        for f in [srv.submit(serving.HullRequest(**scene_args(pool[i % pool_size], pool[i % pool_size].masks),
                                                 blur=pool[i % pool_size].blur)) for i in range(workers)]:
            f.result()
        t0 = time.perf_counter()
        for i in range(n):
            t_sched = t0 + float(arrivals[i])
            dt = t_sched - time.perf_counter()
            if dt > 0:
                time.sleep(dt)
            sc = pool[int(picks[i])]
            fut = srv.submit(serving.HullRequest(**scene_args(sc, sc.masks), blur=sc.blur))
            fut.add_done_callback(lambda f, k=int(picks[i]), ts=t_sched: done(f, k, ts))
            del fut
            if (i + 1) % max(1, n // 6) == 0:
                log(f"  submitted {i + 1}/{n}")
        with cv:
            cv.wait_for(lambda: completed[0] >= n)
        t_end = time.perf_counter()
    lat_ms = np.array(lat) * 1e3
    return {"rate_rps": rate, "seconds": seconds, "requests": n, "workers": workers,
            "p50_ms": round(float(np.percentile(lat_ms, 50)), 3), "p99_ms": round(float(np.percentile(lat_ms, 99)), 3),
            "max_ms": round(float(lat_ms.max()), 3), "hulls_per_s": round(n / (t_end - t0), 2),
            "mean_batch": round(float(np.mean(batch_sizes)), 2), "joined_at_level_boundary": joined[0],
            "mismatches_vs_plain": mismatches[0],
            "pool": f"{pool_size} mixed scenes, levels 6-10, 4-48 cameras, 256/512/1024 px, partial p=0.3, blur k7"}


def _cpu_model() -> str:
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return platform.processor() or platform.machine()


def cpu_baseline(scenes, gpu_meshes, budget_s: float) -> dict:
    """The CPU oracle (C++ restatement of the reference path, OpenMP) on a fixed sample of the workload:
    1 warm-up then the median of 5 timed runs on all host threads, and a single-thread figure on the
    sample's first scene (1 warm-up, median of 3).  Wall time from host-resident masks to a host-resident
    mesh (blur, integral, carving, field, marching cubes); every sample mesh is compared with the GPU's."""
    from oracle import oracle

    cores = len(os.sched_getaffinity(0))
    host = [(sc, sc.masks.cpu().numpy(), sc.transforms.cpu().numpy()) for sc in scenes]

    def run(items):
        out = []
        for sc, m, T in items:
            if sc.blur is not None:
                m = oracle.gaussian_blur_sparse(m.astype(np.float64), sc.blur[0], sc.blur[1], np.float32)
            out.append(oracle.visual_hull(m, T, sc.level, sc.cube_corner_bfl, sc.cube_length, sc.masks_partial,
                                          sc.transforms_convention, True))
        return out

    def timed_runs(items, reps):
        t = []
        res = run(items)  # warm-up
        for _ in range(reps):
            t0 = time.perf_counter()
            res = run(items)
            t.append(time.perf_counter() - t0)
        return statistics.median(t), res

    oracle.set_threads(cores)
    # the sample: the first scenes whose single pass fits ~1/7 of the budget (warm-up + 5 runs + 1 thread)
    sample, t_acc = [], 0.0
    for item in host:
        t0 = time.perf_counter()
        run([item])
        t_acc += time.perf_counter() - t0
        sample.append(item)
        if t_acc >= budget_s / 7.0:
            break
    med, res = timed_runs(sample, 5)
    mism = 0
    for (sc, _, _), (v, f), (gv, gf) in zip(sample, res, gpu_meshes):
        gv, gf = gv.cpu().numpy(), gf.cpu().numpy()
        ok = gf.shape == f.shape and np.array_equal(gf, f) and gv.shape == v.shape and \
            np.allclose(gv, v, rtol=0, atol=1e-6 * sc.cube_length, equal_nan=True)
        mism += 0 if ok else 1
    oracle.set_threads(1)
    med1, _ = timed_runs(sample[:1], 3)
    oracle.set_threads(cores)
    desc = ", ".join(f"{s.num_cameras}cam/{s.masks.shape[1]}px/L{s.level}" for s, _, _ in sample)
    return {"value": round(len(sample) / med, 4), "unit": "hulls/s", "cores": cores, "kind": "port",
            "sample": f"first {len(sample)} scenes of the mixed64 workload ({desc}): blur + carve + field + MC, "
                      f"median of 5 runs after 1 warm-up, {med:.2f} s per run on {cores} threads of {_cpu_model()}",
            "median_s": round(med, 3), "runs": 5, "warmup": 1, "cpu_model": _cpu_model(),
            "single_core": {"value": round(1.0 / med1, 4), "unit": "hulls/s", "cores": 1,
                            "sample": "first scene of the sample, median of 3 runs after 1 warm-up",
                            "median_s": round(med1, 3)},
            "oracle_mesh_mismatches": mism, "oracle_scenes_checked": len(sample)}


def measure_c2(dev: torch.device) -> dict:
    """Level-10 carving of config 2 (32 x 2048^2, OpenCV, partial masks, blur k15 sigma 3): its algorithmic
    bytes over its HIP-event time, and the whole hull time.  The blurred masks leave no window that carving
    could skip (solid_reach.h), so every counted camera test is made, with 4 integral reads of 4 B; parents
    and children are read and written once, 4 B each."""
    log("config 2 (32 x 2048^2, level 10, opencv, partial): rendering ...")
    sc2 = synthetic.config_scene(2, 0, device=dev)
    m2 = blur(sc2)
    run2 = lambda: th.visual_hull(**scene_args(sc2, m2), unique_verts=True)  # noqa: E731
    t2, _ = timed(run2, 3, 1)
    p2 = carve_profile(run2)
    last = p2["levels"][-1]
    moved = 4 * last["parents"] + 16 * last["camera_tests"] + 4 * last["children"]
    return {"level": last["level"], "kernel": last["kernel"], "ms": round(last["ms"], 4), "bytes": moved,
            "parents": last["parents"], "camera_tests": last["camera_tests"],
            "achieved_GBs": round(moved / (last["ms"] * 1e-3) / 1e9, 1),
            "frac": round(moved / (last["ms"] * 1e-3) / 1e9 / HBM_PEAK_GBS, 4),
            "camera_tests_per_s": round(last["camera_tests"] / (last["ms"] * 1e-3), 1),
            "hull_ms": round(1e3 * t2 / 3, 3)}


def main() -> None:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--scenes", type=int, default=64)
    ap.add_argument("--cpu-seconds", type=float, default=15.0)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-c2", action="store_true", help="skip the level-10 carving measurement of config 2")
    ap.add_argument("--batched-only", action="store_true", help="skip the per-scene path (for profiling runs)")
    ap.add_argument("--serve-seconds", type=float, default=60.0, help="length of the serving run (0: skip)")
    ap.add_argument("--serve-rate", type=float, default=200.0, help="Poisson request rate of the serving run")
    ap.add_argument("--serve-workers", type=int, default=3)
    ap.add_argument("--serve-loaded-rate", type=float, default=600.0,
                    help="Poisson rate of a second, loaded serving point (0: skip)")
    ap.add_argument("--serve-loaded-seconds", type=float, default=15.0)
    ap.add_argument("--serve-pool", type=int, default=32)
    ap.add_argument("--workload", choices=["mixed64", "c2"], default="mixed64",
                    help="c2: only the config-2 (32 x 2048^2, level 10) measurement, for profiling runs")
    ap.add_argument("--calibrate-copy-mib", type=int, default=0,
                    help="first run one elementwise int32 kernel (bitwise_not) that reads and writes this many MiB "
                         "(HBM counter calibration)")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py: measures one GPU; --gpus {args.gpus} is not supported "
              f"(scenes are independent, so N GPUs would each run their own batch)", flush=True)
        sys.exit(2)
    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)

    if args.calibrate_copy_mib > 0:
        n = args.calibrate_copy_mib * 2**20 // 4
        src = torch.ones(n, dtype=torch.int32, device=dev)
        dst = torch.empty_like(src)
        torch.cuda.synchronize()
        torch.bitwise_not(src, out=dst)  # one elementwise kernel: n * 4 bytes read, n * 4 bytes written
        torch.cuda.synchronize()
        log(f"calibration kernel: {args.calibrate_copy_mib} MiB read + {args.calibrate_copy_mib} MiB written")
        del src, dst

    if args.workload == "c2":
        print(json.dumps({"config2_level10_carve": measure_c2(dev)}), flush=True)
        return

    log("rendering mixed workload scenes on the GPU ...")
    scenes = synthetic.mixed_scenes(args.scenes, device=dev)
    torch.cuda.synchronize()
    mask_bytes = sum(sc.masks.numel() * 4 for sc in scenes)
    log(f"  {len(scenes)} scenes, {mask_bytes / 2**30:.2f} GiB of masks")

    t_h, _ = timed(lambda: step_batched(scenes, graph=False), max(1, args.steps // 2), 1)
    log(f"batched, host-driven carving loop: {1e3 * t_h / max(1, args.steps // 2):.2f} ms/step")
    t_b, meshes_b = timed(lambda: step_batched(scenes), args.steps, args.warmup)
    log(f"batched: {1e3 * t_b / args.steps:.2f} ms/step")
    t_s, mismatch = None, None
    if not args.batched_only:
        t_s, meshes_s = timed(lambda: step_per_scene(scenes), args.steps, args.warmup)
        log(f"per-scene: {1e3 * t_s / args.steps:.2f} ms/step")
        mismatch = 0
        for (vb, fb), (vs, fs) in zip(meshes_b, meshes_s):
            if not (torch.equal(fb, fs) and torch.equal(vb.view(torch.int32), vs.view(torch.int32))):
                mismatch += 1

    prof = carve_profile(lambda: step_batched(scenes))
    roof = roofline_from(prof["levels"])

    result = {
        "metric": "visual hulls/s batched vs per-scene on 1 GPU (exact mesh match) + p50/p99 latency",
        "value": round(len(scenes) * args.steps / t_b, 3),
        "unit": "hulls/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(1e3 * t_b / args.steps, 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic (seeded ellipsoid unions, exact ray-ellipsoid masks rendered on the GPU)",
        "config": {"workload": "mixed64: 64 scenes, 1-8 ellipsoids, 4-48 cameras, 256/512/1024 px, level 6-9, "
                               "masks_partial p=0.3, blur k7 sigma1.5, opengl", "scenes": len(scenes),
                   "mask_gib": round(mask_bytes / 2**30, 3)},
        "per_scene_hulls_per_s": None if t_s is None else round(len(scenes) * args.steps / t_s, 3),
        "batched_over_per_scene": None if t_s is None else round(t_s / t_b, 3),
        "exact_match": {"batched_vs_per_scene_mismatches": mismatch, "scenes": len(scenes)},
        "batched_host_driven_ms_per_step": round(1e3 * t_h / max(1, args.steps // 2), 3),
        "graph_replay": th.graph_stats(dev),
        "roofline": roof,
        "carve_levels": prof["levels"],
    }

    if not args.no_c2:
        result["config2_level10_carve"] = measure_c2(dev)

    if args.serve_seconds > 0:
        result["serving"] = serve(args.serve_rate, args.serve_seconds, args.serve_pool, args.serve_workers, dev)
        if args.serve_loaded_rate > 0:
            result["serving_loaded"] = serve(args.serve_loaded_rate, args.serve_loaded_seconds, args.serve_pool,
                                             args.serve_workers, dev)

    if not args.no_cpu_baseline:
        log("CPU baseline (oracle) ...")
        result["cpu_baseline"] = cpu_baseline(scenes, meshes_b, args.cpu_seconds)
    print(json.dumps(result), flush=True)


if __name__ == "__main__":
    main()
