"""Performance cases of the framework: what its users have it do, through its public entry points.

listed()              the named cases, each with a comment on what it stands for
draw(rng)             one more case of the same ranges
prepare(case, seed)   what a program holds before the call: masks and cameras, or a volume, on the GPU
run(state)            one pass through the public entry points, and its outputs
work(case)            bytes and operations that one pass cannot do without
exact(case, seed)     the floating-point outputs in 64 bits, where their layout does not hang on rounding

Scenes are unions of ellipsoids seen by pinhole cameras around them (torchhull_amd.synthetic), rendered on the
GPU: silhouettes with the size, the share of the image and the smooth outline that segmentation masks of an
object in a camera ring have. Volumes are signed distances to unions of spheres. The geometry belongs to the
case, so that a mesh has the same size for every seed: the seed mirrors and scales a scene (by signs and powers
of two, which carry through every rounding) and swaps its first two cameras, it bends a volume by a smooth
positive factor, and it draws the images of a blur anew. The sizes are those of the workloads in
torchhull_amd/synthetic.py and of the reference's benchmarks (visual hulls of levels 7-11 from 10-50 cameras at
1920 x 1080, marching cubes of 100^3 to 600^3, blurs of 10-50 masks with kernels of 3-11).
"""

from __future__ import annotations

import math
import random

import numpy as np
import torch

import torchhull_amd as th
from torchhull_amd import synthetic

DEVICE = "cuda"

_DTYPES = {"f16": torch.float16, "f32": torch.float32, "f64": torch.float64, "u8": torch.uint8, "bool": torch.bool}
_BYTES = {"f16": 2, "f32": 4, "f64": 8, "u8": 1, "bool": 1}


def listed() -> list[dict]:
    return [
        # The smallest interactive call: a coarse preview of one object from a small ring of low-resolution masks.
        dict(name="hull_preview_l7", scene=1, kind="hull", level=7, cameras=8, height=256, width=256, dtype="f32",
             blur=0, sigma=1.0, partial=False, convention="opengl", unique=True, output="mesh"),
        # Full-HD capture with 8-bit masks as a segmentation writes them, no blur: the ordinary per-frame hull.
        dict(name="hull_hd_u8_l8", scene=2, kind="hull", level=8, cameras=10, height=1080, width=1920, dtype="u8",
             blur=0, sigma=1.0, partial=False, convention="opengl", unique=True, output="mesh"),
        # A dense camera dome with antialiased masks: blur and hull, the pipeline for a smooth mesh.
        dict(name="hull_dome_blur_l9", scene=3, kind="hull", level=9, cameras=64, height=1024, width=1024, dtype="f32",
             blur=9, sigma=2.0, partial=False, convention="opengl", unique=True, output="mesh"),
        # Close-up cameras that see only parts of the object (partial masks), calibrated in the OpenCV convention.
        dict(name="hull_partial_cv_l10", scene=4, kind="hull", level=10, cameras=32, height=2048, width=2048,
             dtype="f32", blur=15, sigma=3.0, partial=True, convention="opencv", unique=True, output="mesh"),
        # The finest hull of the reference's benchmark: offline reconstruction from 50 Full-HD cameras.
        dict(name="hull_offline_l11", scene=5, kind="hull", level=11, cameras=50, height=1080, width=1920, dtype="f32",
             blur=0, sigma=1.0, partial=False, convention="opengl", unique=True, output="mesh"),
        # The sparse field for a program that extracts or optimises the surface itself; boolean masks of an odd size.
        dict(name="field_bool_odd_l8", scene=6, kind="hull", level=8, cameras=17, height=719, width=1277, dtype="bool",
             blur=0, sigma=1.0, partial=True, convention="opencv", unique=True, output="field"),
        # Many independent scenes at once (a data set, a serving batch): mixed cameras, resolutions and levels.
        dict(name="batch_mixed_24", kind="batch", scenes=24, mix=3000, max_level=9, blur=7, sigma=1.5, unique=True),
        # A dense distance volume of a reconstruction grid, as large as the reference's benchmark goes in earnest.
        dict(name="mc_dense_500", scene=7, kind="mc", layout="dense", depth=500, height=500, width=500, dtype="f32",
             local=True, unique=True, spheres=1),
        # A small non-cubic volume in double precision: an inner step of an optimisation, bound by latency.
        dict(name="mc_dense_f64_small", scene=8, kind="mc", layout="dense", depth=61, height=83, width=71, dtype="f64",
             local=False, unique=True, spheres=3),
        # The narrow band of a distance field as a sparse COO tensor.
        dict(name="mc_sparse_400", scene=9, kind="mc", layout="sparse", depth=400, height=400, width=400, dtype="f32",
             local=True, unique=True, spheres=1),
        # Antialiasing of a capture's binary masks ahead of the hull: the band blur.
        dict(name="blur_band_hd_k7", kind="blur", cameras=30, height=1080, width=1920, dtype="f32", out="f32",
             kernel=7, sigma=1.0, sparse=True),
        # The dense blur (every pixel), the alternative for masks that are not piecewise constant.
        dict(name="blur_dense_hd_k11", kind="blur", cameras=10, height=1080, width=1920, dtype="f32", out="f32",
             kernel=11, sigma=1.0, sparse=False),
    ]


def _log_uniform(rng: random.Random, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["hull", "hull", "hull", "batch", "mc", "mc", "blur", "blur"])
    if kind == "hull":
        level = rng.randint(5, 11)
        height, width = _log_uniform(rng, 120, 2048), _log_uniform(rng, 120, 2048)
        cameras = min(_log_uniform(rng, 4, 64), 120_000_000 // (height * width))
        case = dict(kind="hull", scene=rng.randrange(1 << 30), level=level, cameras=cameras, height=height,
                    width=width, dtype=rng.choice(["f32", "f32", "u8", "bool"]),
                    blur=rng.choice([0, 0, 3, 5, 7, 9, 11, 15]), sigma=round(rng.uniform(0.8, 3.0), 3),
                    partial=rng.random() < 0.3, convention=rng.choice(["opengl", "opencv"]),
                    unique=rng.random() < 0.8, output=rng.choice(["mesh", "mesh", "mesh", "field", "candidates"]))
        if level == 11:  # the listed case of this level is the costliest
            case.update(cameras=min(cameras, 40, 60_000_000 // (height * width)), blur=0, partial=False, unique=True,
                        output="mesh")
        return case
    if kind == "batch":
        return dict(kind="batch", scenes=_log_uniform(rng, 2, 32), mix=rng.randrange(1 << 30),
                    max_level=rng.randint(7, 9), blur=rng.choice([5, 7, 9]), sigma=round(rng.uniform(0.8, 2.5), 3),
                    unique=True)
    if kind == "mc":
        layout = rng.choice(["dense", "sparse"])
        size = _log_uniform(rng, 20, 500)
        dims = [max(8, min(500, int(size * rng.uniform(0.7, 1.3)))) for _ in range(3)]
        return dict(kind="mc", scene=rng.randrange(1 << 30), layout=layout, depth=dims[0], height=dims[1],
                    width=dims[2], dtype=rng.choice(["f32", "f32", "f64"]), local=rng.random() < 0.5,
                    unique=rng.random() < 0.8, spheres=rng.randint(1, 4))
    return dict(kind="blur", cameras=_log_uniform(rng, 1, 50), height=_log_uniform(rng, 64, 1440),
                width=_log_uniform(rng, 64, 1920), dtype=rng.choice(["f32", "f32", "u8", "bool"]),
                out=rng.choice(["f32", "f32", "f32", "f16", "f64"]), kernel=rng.choice([3, 5, 7, 9, 11, 15]),
                sigma=round(rng.uniform(0.8, 3.0), 3), sparse=rng.random() < 0.7)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------


def _scene(seed: int, cameras: int, height: int, width: int, dtype: str, partial: bool, convention: str,
           ellipsoids: int) -> tuple[torch.Tensor, torch.Tensor]:
    """Masks [B,H,W,1] and transforms [B,4,4] of one scene in the cube [-1, 1]^3."""
    rng = np.random.default_rng(seed)
    centers = rng.uniform(-0.4, 0.4, size=(ellipsoids, 3))
    axes = rng.uniform(0.15, 0.4, size=(ellipsoids, 3))
    rotations = [synthetic.random_rotation(rng) for _ in range(ellipsoids)]
    # partial: cameras close enough that parts of the object leave the image
    radius, fovy = (1.6, math.radians(60.0)) if partial else (2.5, math.radians(40.0))
    # `fovy` spans the shorter side, so that the object keeps its share of narrow images too
    if width < height:
        fovy = 2.0 * math.atan(math.tan(fovy / 2.0) * height / width)
    views = np.stack([synthetic.look_at(e) for e in synthetic.fibonacci_cameras(cameras, radius)])
    masks = synthetic.render_masks_gl(views, fovy, height, width, centers, np.stack(rotations), axes, device=DEVICE)
    if convention == "opengl":
        T = np.einsum("ij,bjk->bik", synthetic.perspective(fovy, width / height, 0.1, 1000.0), views)
    else:
        D = np.diag([1.0, -1.0, -1.0, 1.0])
        P = synthetic.perspective_cv(fovy, width / height, height, width)
        T = np.einsum("ij,bjk->bik", P, np.einsum("ij,bjk,kl->bil", D, views, D))
        masks = masks.flip(1)
    return masks.to(_DTYPES[dtype]).contiguous(), torch.as_tensor(T.astype(np.float32), device=DEVICE)


def _posed(masks: torch.Tensor, transforms: torch.Tensor, seed: int) -> dict:
    """The scene mirrored along the axes, scaled, and its first two cameras swapped, as the seed says: the hull is
    the mirrored and scaled one, bit for bit, since signs and powers of two pass through every rounding."""
    scale = 2.0 ** ((seed // 8) % 7 - 3)
    pose = [(-1.0 if seed >> a & 1 else 1.0) / scale for a in range(3)] + [1.0]
    transforms = transforms * torch.tensor(pose, dtype=torch.float32, device=transforms.device)
    if (seed // 56) % 2:
        order = [1, 0] + list(range(2, masks.shape[0]))
        masks, transforms = masks[order].contiguous(), transforms[order].contiguous()
    return dict(masks=masks, transforms=transforms.contiguous(), corner=(-scale, -scale, -scale), length=2.0 * scale)


def _mixed_specs(case: dict) -> list[synthetic.SceneSpec]:
    """The scene shapes of a batch: part of the case, so that every seed has the same ones."""
    rng = np.random.default_rng(case["mix"])
    return [synthetic.mixed_spec(rng, max_level=case["max_level"]) for _ in range(case["scenes"])]


def _volume(case: dict, seed: int) -> torch.Tensor:
    """Signed distance to a union of spheres on a [1,D,H,W] grid, in voxels, zero beyond the band of a sparse
    volume; its zero level is the case's, the slope there the seed's."""
    rng = np.random.default_rng(case["scene"])
    dims = (case["depth"], case["height"], case["width"])
    dtype = _DTYPES[case["dtype"]]
    n = case["spheres"]
    half = 0.5 * min(dims)
    out = None
    for _ in range(n):
        # one sphere fills the grid, several share it
        r = half * (rng.uniform(0.8, 0.9) if n == 1 else rng.uniform(0.35, 0.6))
        c = [rng.uniform(0.5 * (d - 1) - 0.05 * half, 0.5 * (d - 1) + 0.05 * half) if n == 1
             else rng.uniform(r + 1.0, max(r + 1.0, d - r - 2.0)) for d in dims]
        g = [(torch.arange(d, dtype=torch.float64, device=DEVICE) - m) ** 2 for d, m in zip(dims, c)]
        sq = (g[0].view(-1, 1, 1) + g[1].view(1, -1, 1)) + g[2].view(1, 1, -1)
        dist = (sq.sqrt_() - r).to(dtype)
        out = dist if out is None else torch.minimum(out, dist)
    if case["layout"] == "sparse":
        out[out.abs() > 2] = 0
    rng = np.random.default_rng(seed)
    for axis, d in enumerate(dims):  # a positive factor between 0.51 and 1.73
        phase, waves = rng.uniform(0.0, 2.0 * math.pi), rng.uniform(1.0, 3.0)
        t = torch.arange(d, dtype=torch.float64, device=DEVICE) * (2.0 * math.pi * waves / d) + phase
        out *= (1.0 + 0.2 * torch.sin(t) * (1 if axis else -1)).to(dtype).view(
            [-1 if a == axis else 1 for a in range(3)])
    return out.unsqueeze(0).contiguous()


def prepare(case: dict, seed: int) -> dict:
    if case["kind"] == "hull":
        masks, transforms = _scene(case["scene"], case["cameras"], case["height"], case["width"], case["dtype"],
                                   case["partial"], case["convention"], 6)
        return dict(case=case, **_posed(masks, transforms, seed))
    if case["kind"] == "batch":
        scenes = []
        for i, spec in enumerate(_mixed_specs(case)):
            m, T = _scene(case["mix"] + i, spec.n_cameras, spec.resolution, spec.resolution, "f32",
                          spec.masks_partial, spec.convention, spec.n_ellipsoids)
            p = _posed(m, T, seed + i)
            scenes.append(dict(masks=p["masks"], transforms=p["transforms"], level=spec.level,
                               cube_corner_bfl=p["corner"], cube_length=p["length"],
                               masks_partial=spec.masks_partial, transforms_convention=spec.convention))
        return dict(case=case, scenes=scenes)
    if case["kind"] == "mc":
        volume = _volume(case, seed)
        if case["layout"] == "sparse":
            volume = volume.to_sparse()
        return dict(case=case, volume=volume)
    masks, _ = _scene(seed, case["cameras"], case["height"], case["width"], case["dtype"], False, "opengl", 6)
    return dict(case=case, images=masks)


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------


def run(state: dict):
    case = state["case"]
    if case["kind"] == "hull":
        masks = state["masks"]
        if case["blur"]:
            masks = th.gaussian_blur(masks, case["blur"], case["sigma"], sparse=True, dtype=torch.float32)
        args = (masks, state["transforms"], case["level"], state["corner"], state["length"], case["partial"],
                case["convention"])
        if case["output"] == "field":
            field = th.sparse_visual_hull_field(*args)
            return field.indices(), field.values()
        if case["output"] == "candidates":
            return th.visual_hull_with_candidate_voxels(*args, unique_verts=case["unique"])
        return th.visual_hull(*args, unique_verts=case["unique"])
    if case["kind"] == "batch":
        scenes = state["scenes"]
        blurred = th.gaussian_blur_batch([s["masks"] for s in scenes], case["blur"], case["sigma"], sparse=True,
                                         dtype=torch.float32)
        return th.visual_hull_batch([dict(s, masks=m) for s, m in zip(scenes, blurred)], unique_verts=case["unique"])
    if case["kind"] == "mc":
        return th.marching_cubes(state["volume"], 0.0, return_local_coords=case["local"],
                                 unique_verts=case["unique"])
    return th.gaussian_blur(state["images"], case["kernel"], case["sigma"], sparse=case["sparse"],
                            dtype=_DTYPES[case["out"]])


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------


def _hull_work(cameras: int, height: int, width: int, elem: int, level: int, mesh: bool, unique: bool) -> tuple:
    # The hull's surface in units of finest cells: about 4 area units in a cube of side 2, so 4^level cells;
    # 1.5 grid edges and 3 triangles cross per cell (about 3.3 field vertices per cell).
    cells = 4.0 ** level
    if mesh:
        out = cells * ((1.5 if unique else 9.0) * 12 + 3 * 24)
    else:
        out = 3.3 * cells * (4 * 8 + 4)
    # Every kept cell of every level was classified with its 7 siblings in its cameras (about 30 operations a
    # test with shared corners), and every field vertex sampled in every camera (about 50 operations).
    flops = cameras * cells * (4.0 / 3.0 * 2.0 * 30 + 3.3 * 50)
    return cameras * height * width * elem + out, flops


def work(case: dict) -> dict:
    if case["kind"] == "hull":
        b, f = _hull_work(case["cameras"], case["height"], case["width"], _BYTES[case["dtype"]], case["level"],
                          case["output"] != "field", case["unique"])
        return {"bytes": b, "flops": f}
    if case["kind"] == "batch":
        parts = [_hull_work(s.n_cameras, s.resolution, s.resolution, 4, s.level, True, case["unique"])
                 for s in _mixed_specs(case)]
        return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}
    if case["kind"] == "mc":
        elem = _BYTES[case["dtype"]]
        dims = (case["depth"], case["height"], case["width"])
        area = math.pi * (0.85 * min(dims)) ** 2  # voxels that the surface passes through, about 1.5 per unit
        voxels = dims[0] * dims[1] * dims[2]
        read = voxels * elem if case["layout"] == "dense" else 4.0 * area * (4 * 8 + elem)
        cells = voxels if case["layout"] == "dense" else 4.0 * area
        return {"bytes": read + area * ((1.5 if case["unique"] else 9.0) * 12 + 3 * 24),
                "flops": 8.0 * cells + 1.5 * area * 10}
    pixels = case["cameras"] * case["height"] * case["width"]
    taps = 2.0 * case["kernel"] ** 2
    # the band covers about a tenth of the pixels per 10 columns of the kernel at most
    share = 1.0 if not case["sparse"] else 0.01 * case["kernel"]
    return {"bytes": pixels * (_BYTES[case["dtype"]] + _BYTES[case["out"]]), "flops": pixels * (2 + taps * share)}


# ---------------------------------------------------------------------------
# Results in 64 bits
# ---------------------------------------------------------------------------


def _shifted(t: torch.Tensor, off: tuple[int, int, int], fill) -> torch.Tensor:
    """t moved so that element (z, y, x) holds t[z + off_z, y + off_y, x + off_x], `fill` outside."""
    out = torch.full_like(t, fill)
    dst = tuple(slice(max(0, -o), t.shape[a] - max(0, o)) for a, o in enumerate(off))
    src = tuple(slice(max(0, o), t.shape[a] - max(0, -o)) for a, o in enumerate(off))
    out[dst] = t[src]
    return out


def _exact_mc_vertices(case: dict, seed: int) -> torch.Tensor:
    """Vertices of the compact mesh: the sign-changing grid edges next to a complete cell, in the order of
    (z, y, x) of the lower endpoint, then of the axis x, y, z."""
    volume = _volume(case, seed)[0]
    present = volume != 0 if case["layout"] == "sparse" else torch.ones_like(volume, dtype=torch.bool)
    complete = present.clone()
    for dz in (0, 1):
        for dy in (0, 1):
            for dx in (0, 1):
                complete &= _shifted(present, (dz, dy, dx), False)
    units = {0: (0, 0, 1), 1: (0, 1, 0), 2: (1, 0, 0)}  # axis x, y, z
    below = volume < 0
    emitted = []
    for axis in range(3):
        e = present & _shifted(present, units[axis], False) & (below != _shifted(below, units[axis], False))
        a, b = (units[q] for q in range(3) if q != axis)
        near = complete.clone()
        for u in ((-a[0], -a[1], -a[2]), (-b[0], -b[1], -b[2]), (-a[0] - b[0], -a[1] - b[1], -a[2] - b[2])):
            near |= _shifted(complete, u, False)
        emitted.append(e & near)
    at = torch.stack(emitted, dim=-1).nonzero()  # (z, y, x, axis) in ascending order
    del emitted, complete, present, below
    lower, axis = at[:, :3], at[:, 3]
    step = torch.tensor([units[q] for q in range(3)], device=at.device)[axis]
    upper = lower + step
    v1 = volume[lower[:, 0], lower[:, 1], lower[:, 2]].double()
    v2 = volume[upper[:, 0], upper[:, 1], upper[:, 2]].double()
    eps = 1e-5  # values this near to the level, or to each other, snap to an endpoint
    t = -v1 / (v2 - v1)
    t = torch.where((v1 - v2).abs() < eps, torch.zeros_like(t), t)
    t = torch.where(v2.abs() < eps, torch.ones_like(t), t)
    t = torch.where(v1.abs() < eps, torch.zeros_like(t), t)
    p = (lower.double() + t[:, None] * step.double()).flip(1)  # x, y, z
    if case["local"]:
        size = torch.tensor([case["width"], case["height"], case["depth"]], dtype=torch.float64, device=p.device)
        p = p * (2.0 / (size - 1.0)) - 1.0
    return p


def _exact_blur(case: dict, seed: int) -> torch.Tensor:
    images = prepare(case, seed)["images"][..., 0]
    B, H, W = images.shape
    k, h = case["kernel"], case["kernel"] // 2
    off = range(-h, h + 1)
    weights = {(i, j): math.exp(-(i * i + j * j) / (2.0 * case["sigma"] ** 2)) for i in off for j in off}
    total = math.fsum(weights.values())
    out = torch.empty((B, H, W, 1), dtype=torch.float64, device=images.device)
    for b in range(B):
        src = images[b].double()
        pad = torch.nn.functional.pad(src[None, None], (h, h, h, h), mode="reflect")[0, 0]
        acc = torch.zeros_like(src)
        for (i, j), w in weights.items():  # i: columns, j: rows
            acc += w * pad[h + j:h + j + H, h + i:h + i + W]
        acc /= total
        if case["sparse"]:
            # pixels that differ from their right or lower neighbour, spread over the 3 x 3 tiles around theirs
            edge = torch.zeros((H, W), dtype=torch.bool, device=src.device)
            edge[:, :-1] |= src[:, 1:] != src[:, :-1]
            edge[:-1, :] |= src[1:, :] != src[:-1, :]
            rows = torch.arange(H, device=src.device) // h
            cols = torch.arange(W, device=src.device) // h
            tiles = torch.zeros((H // h + 1, W // h + 1), dtype=torch.float64, device=src.device)
            at = edge.nonzero()
            tiles[rows[at[:, 0]], cols[at[:, 1]]] = 1.0
            band = torch.nn.functional.max_pool2d(tiles[None, None], 3, stride=1, padding=1)[0, 0] > 0
            acc = torch.where(band[rows][:, cols], acc, src)
        out[b, :, :, 0] = acc
    return out


def exact(case: dict, seed: int):
    # Hulls: which cells are kept hangs on the rounding of pixel windows, so their vertices have no layout in 64 bits.
    if case["kind"] == "mc" and case["unique"]:
        return _exact_mc_vertices(case, seed), None
    if case["kind"] == "blur":
        return _exact_blur(case, seed)
    return None
