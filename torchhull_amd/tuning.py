"""Autotuner of the carving launch shape (lanes per parent by octree level size).

Carving classifies each level in one launch.  Small levels split a parent's
cameras over G lanes (64, 16, 4 or 2) to fill the GPU; large ones use one lane per
parent.  Which G is fastest for a level of n parents depends on the device and
on the scenes (cameras per scene, early exits), so it is measured:
`tune_carving` runs each workload once per G with that G's threshold forced on every
level and reads every level's classification time (HIP events,
`thull_profile_carve`).  What it measures is what the threshold stands for: of the
levels that ask for 64 lanes the library gives the smallest a kernel of their own
and scenes of few cameras fewer lanes (`split_for` with `cameras`).  It then picks
the four level-size thresholds that minimise the sum of all measured levels, each
as a share of its workload's whole call, so that a preview counts as much as a
level-11 hull.  Present thresholds stay where they cost next to nothing (SLACK); a
new one lies half way (by the logarithm) between the measured sizes around it.  The choice never changes a result, only its speed.

`python -m torchhull_amd.tuning --out torchhull_amd/carve_tuning.json` tunes on
`workloads(seed)`: single hulls of levels 6 to 11 and mixed batches, drawn over the
range of cameras, image sizes, conventions and blurs, every other batch as a replayed
loop; checks the choice on another draw of them; and writes the thresholds, which
`_lib.context` applies to every new context when the file is there.
"""

from __future__ import annotations

import argparse
import ctypes
import json
import math
import pathlib
import statistics
import time
from typing import Callable, Iterator, Sequence

import numpy as np
import torch

from . import _lib

DEFAULT_PATH = pathlib.Path(__file__).resolve().parent / "carve_tuning.json"
_MAX = 0xFFFFFFFF
_N = 4  # thresholds: G = 64, 16, 4, 2 up to max_parents[0..3], else 1
# thresholds that force one G on every level
_FORCE = {64: (_MAX,) * 4, 16: (0,) + (_MAX,) * 3, 4: (0, 0, _MAX, _MAX), 2: (0, 0, 0, _MAX), 1: (0,) * 4}


def set_carve_tuning(ctx: ctypes.c_void_p, max_parents: Sequence[int]) -> None:
    arr = (ctypes.c_uint32 * _N)(*[int(v) for v in max_parents])
    _lib.check(_lib.lib().thull_ctx_set_carve_tuning(ctx, arr))


def get_carve_tuning(ctx: ctypes.c_void_p) -> list[int]:
    arr = (ctypes.c_uint32 * _N)()
    _lib.check(_lib.lib().thull_ctx_get_carve_tuning(ctx, arr))
    return list(arr)


def split_for(n: int, max_parents: Sequence[int], cameras: int | None = None) -> int:
    """Lanes per parent that the thresholds ask for at a level of n parents (the library's
    carve_split_factor): G falls back to fewer lanes while n * G would not fit 31 bits.  With the most
    `cameras` of a scene, the kernel that the library launches for it: 8 stands for the kernel of the
    smallest levels, and lanes that the cameras would leave idle are not used (launch_carve_classify)."""
    g = 1
    if n <= max_parents[0]:
        g = 64
    elif n <= max_parents[1]:
        g = 16
    elif n <= max_parents[2]:
        g = 4
    elif n <= max_parents[3]:
        g = 2
    while g > 1 and n * g >= 1 << 31:
        g = {64: 16, 16: 4, 4: 2, 2: 1}[g]
    if cameras is None:
        return g
    if g == 64:
        group = 8
        while group < min(cameras, 64):
            group *= 2
        if n * group // 8 <= 8192:
            return 8
        if cameras <= 16:
            g = 16
    return 4 if g == 16 and cameras <= 4 else g


def measure_levels(run: Callable[[], object], ctx: ctypes.c_void_p, reps: int = 3) -> list[tuple[int, float]]:
    """(parents, median classification ms) of every carving step of run()."""
    L = _lib.lib()
    n = 16
    runs = []
    for _ in range(reps):
        _lib.check(L.thull_profile_enable(ctx, 1))
        try:
            run()
            torch.cuda.synchronize()
        finally:
            _lib.check(L.thull_profile_enable(ctx, 0))
        ms = (ctypes.c_float * n)()
        par, tests, nxt = (ctypes.c_int64 * n)(), (ctypes.c_int64 * n)(), (ctypes.c_int64 * n)()
        split = (ctypes.c_int32 * n)()
        _lib.check(L.thull_profile_carve(ctx, n, ms, par, tests, nxt, split))
        runs.append([(int(par[i]), float(ms[i])) for i in range(n) if par[i] > 0])
    return [(runs[0][i][0], statistics.median(r[i][1] for r in runs)) for i in range(len(runs[0]))]


def _between(lo: int, hi: int) -> int:
    """A threshold in [lo, hi): half way by the logarithm, to two digits where that fits."""
    t = int(math.sqrt(lo * hi))
    digit = 10 ** max(0, len(str(t)) - 2)
    rounded = (t + digit // 2) // digit * digit
    return rounded if lo <= rounded < hi else t


# A choice between thresholds whose costs differ by less than this is the draw's, not the device's (the own
# thresholds of another draw gain 0.2 % on it): the present ones stay.
SLACK = 0.002


def choose_thresholds(samples: dict[int, list[tuple[int, float]]], weights: Sequence[float] | None = None,
                      present: Sequence[int] | None = None) -> tuple[list[int], float]:
    """Thresholds minimising the summed (weighted) level time; samples[G] = [(parents, ms), ...] over the same
    levels.  G may only fall as levels grow, so the sizes are cut into five runs: a dynamic program over the cuts.
    Of the `present` thresholds, those stay that leave the sum within SLACK of the least, from the last on."""
    levels = [n for n, _ in samples[1]]
    weights = [1.0] * len(levels) if weights is None else weights
    sizes = sorted(set(levels))
    order = [64, 16, 4, 2, 1]
    cost = []  # [G][size]
    for g in order:
        row = dict.fromkeys(sizes, 0.0)
        for i, n in enumerate(levels):
            row[n] += weights[i] * samples[split_for(n, _FORCE[g])][i][1]
        cost.append([row[n] for n in sizes])
    # best[k]: least cost of the first k sizes with the G so far; cuts[q][k]: how many of them go to earlier ones
    best = [0.0] + [math.inf] * len(sizes)
    cuts = []
    for row in cost:
        new, cut = list(best), list(range(len(sizes) + 1))
        for k in range(1, len(sizes) + 1):
            if new[k - 1] + row[k - 1] < new[k]:
                new[k], cut[k] = new[k - 1] + row[k - 1], cut[k - 1]
        best = new
        cuts.append(cut)
    at, chosen = len(sizes), []
    for cut in reversed(cuts[1:]):
        at = cut[at]
        chosen.append(0 if at == 0 else _MAX if at == len(sizes) else _between(sizes[at - 1], sizes[at]))
    chosen, least = chosen[::-1], best[-1]
    total = least
    for q in reversed(range(_N if present is not None else 0)):
        trial = chosen[:q] + [present[q]] + chosen[q + 1:]
        cost_trial = _shares(samples, weights, trial)
        if trial == sorted(trial) and cost_trial <= least * (1.0 + SLACK):
            chosen, total = trial, cost_trial
    return chosen, total


def _shares(samples: dict[int, list[tuple[int, float]]], weights: Sequence[float], max_parents: Sequence[int]) -> float:
    return sum(w * samples[split_for(n, max_parents)][i][1]
               for i, ((n, _), w) in enumerate(zip(samples[1], weights)))


def measure(runs: Sequence[Callable[[], object]], device_index: int = 0,
            reps: int = 3) -> tuple[dict[int, list[tuple[int, float]]], list[float]]:
    """Level times of every run with every G forced, and each level's weight: 1 / its run's time (ms)."""
    ctx = _lib.context(device_index)
    saved = get_carve_tuning(ctx)
    samples: dict[int, list[tuple[int, float]]] = {g: [] for g in _FORCE}
    weights: list[float] = []
    try:
        for run in runs:
            times = []
            for _ in range(reps + 2):  # the first ones warm up (pool growth, weights)
                torch.cuda.synchronize()
                t0 = time.perf_counter()
                run()
                torch.cuda.synchronize()
                times.append(1e3 * (time.perf_counter() - t0))
            for g, force in _FORCE.items():
                set_carve_tuning(ctx, force)
                _lib.check(_lib.lib().thull_ctx_trim(ctx))
                run()  # a replayed batch plans its loop with this G
                samples[g].extend(measure_levels(run, ctx, reps))
            set_carve_tuning(ctx, saved)
            _lib.check(_lib.lib().thull_ctx_trim(ctx))
            weights += [1.0 / statistics.median(times[2:])] * (len(samples[1]) - len(weights))
    finally:
        set_carve_tuning(ctx, saved)
    return samples, weights


def tune_carving(workloads: Sequence[Callable[[], object]], device_index: int = 0, reps: int = 3) -> dict:
    """Measures every G on every workload and returns the chosen thresholds with the measurements: `shares`
    is the sum over levels of classification time / the workload's call, `default_shares` that of the
    context's present thresholds."""
    saved = get_carve_tuning(_lib.context(device_index))
    samples, weights = measure(workloads, device_index, reps)
    chosen, _ = choose_thresholds(samples, weights, saved)
    return {"max_parents": chosen, "shares": round(_shares(samples, weights, chosen), 4),
            "default_shares": round(_shares(samples, weights, saved), 4),
            "levels": [{"parents": n, "weight": round(weights[i], 4),
                        **{f"ms_g{g}": round(samples[g][i][1], 4) for g in _FORCE}}
                       for i, (n, _) in enumerate(samples[1])]}


def load(path: pathlib.Path = DEFAULT_PATH) -> list[int] | None:
    """Stored thresholds, or None when there is no usable file."""
    try:
        with open(path) as f:
            v = json.load(f)["max_parents"]
        if len(v) == _N and all(isinstance(x, int) and 0 <= x <= _MAX for x in v) and v == sorted(v):
            return v
    except (OSError, ValueError, KeyError, TypeError):
        pass
    return None


def workloads(seed: int, device: torch.device, singles: int = 288,
              batches: int = 36) -> Iterator[tuple[str, Callable[[], object]]]:
    """Single hulls over levels 6 to 11, 4 to 64 cameras and 192 to 2048 pixels, and batches of 2 to 64 mixed scenes."""
    from . import api, synthetic

    rng = np.random.default_rng(seed)

    def log_uniform(lo: float, hi: float) -> int:
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def args(sc: synthetic.Scene, masks: torch.Tensor) -> dict:
        return dict(masks=masks, transforms=sc.transforms, level=sc.level, cube_corner_bfl=sc.cube_corner_bfl,
                    cube_length=sc.cube_length, masks_partial=sc.masks_partial,
                    transforms_convention=sc.transforms_convention)

    for i in range(singles):
        level, partial = 6 + i % 6, bool(rng.random() < 0.3)
        spec = synthetic.SceneSpec(
            n_ellipsoids=int(rng.integers(1, 9)), n_cameras=int(rng.integers(4, 65 if level < 11 else 41)),
            resolution=log_uniform(192, 2048), level=level, masks_partial=partial,
            convention="opencv" if rng.random() < 0.5 else "opengl",
            blur=None if rng.random() < 0.5 else (int(rng.choice([3, 7, 11])), 1.5),
            radius=1.6 if partial else 2.5, fovy_deg=60.0 if partial else 40.0)
        sc = synthetic.make_scene(spec, int(rng.integers(1 << 30)), device=device)
        m = sc.masks if sc.blur is None else api.gaussian_blur(sc.masks, *sc.blur, sparse=True, dtype=torch.float32)
        yield (f"level {level}, {spec.n_cameras} x {spec.resolution}^2{' partial' if partial else ''}",
               lambda a=args(sc, m): api.visual_hull(**a))
    for i in range(batches):
        n, top, graph = log_uniform(2, 64), int(rng.integers(7, 10)), i % 2 == 1
        scenes = synthetic.mixed_scenes(n, seed=int(rng.integers(1 << 30)), device=device, max_level=top)
        blurred = api.gaussian_blur_batch([sc.masks for sc in scenes], *scenes[0].blur, sparse=True,
                                          dtype=torch.float32)
        yield (f"{n} mixed scenes up to level {top}{', replayed' if graph else ''}",
               lambda b=[args(sc, m) for sc, m in zip(scenes, blurred)], g=graph: api.visual_hull_batch(b, graph=g))


def main() -> None:
    ap = argparse.ArgumentParser(description=__doc__.split("\n\n")[0])
    ap.add_argument("--out", type=pathlib.Path, default=DEFAULT_PATH)
    ap.add_argument("--seed", type=int, default=5000)
    ap.add_argument("--reps", type=int, default=3)
    ap.add_argument("--samples", type=pathlib.Path, help="also write every level's times")
    opts = ap.parse_args()
    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    t0 = time.perf_counter()
    runs = []
    for name, run in workloads(opts.seed, dev):
        print(name, flush=True)
        runs.append(run)
    n = len(runs)
    res = tune_carving(runs, reps=opts.reps)
    if opts.samples is not None:
        opts.samples.write_text(json.dumps(res["levels"], indent=1))
    print(json.dumps({k: v for k, v in res.items() if k != "levels"}), flush=True)
    # the choice on workloads that it has not seen
    del runs, run
    saved = get_carve_tuning(_lib.context(0))
    samples, weights = measure([run for _, run in workloads(opts.seed + 1, dev)], reps=opts.reps)
    best, _ = choose_thresholds(samples, weights)
    check = {"max_parents": best, "shares": round(_shares(samples, weights, res["max_parents"]), 4),
             "default_shares": round(_shares(samples, weights, saved), 4),
             "own_shares": round(_shares(samples, weights, best), 4)}
    record = {"max_parents": res["max_parents"],
              "objective": "sum over levels of classification time / the workload's call", "seed": opts.seed,
              "shares": res["shares"], "default_shares": res["default_shares"], "default": list(saved),
              "other_draw": check, "workloads": n, "device": torch.cuda.get_device_name(dev),
              "seconds": round(time.perf_counter() - t0, 1)}
    opts.out.write_text(json.dumps(record, indent=1) + "\n")
    print(json.dumps(record), flush=True)


if __name__ == "__main__":
    main()
