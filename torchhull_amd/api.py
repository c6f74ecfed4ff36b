"""Python entry points, mirroring the reference's bindings (src/torchhull/_C/python/bindings.cpp).

Argument checks raise RuntimeError with the reference's conditions
(visual_hull_cuda.cu:591-613, marching_cubes_cuda.cu:382-385,715-719,762-768,
gaussian_blur_cuda.cu:79-81,294-305).  Tensor plumbing (dtype conversion,
contiguity, output allocation) uses torch; all computation runs in the HIP
library.
"""

from __future__ import annotations

import ctypes
import math
import pathlib
import time
from collections.abc import Sequence

import torch

from . import _lib

_DTYPE_CODES = {
    torch.bool: _lib.BOOL,
    torch.uint8: _lib.U8,
    torch.int8: _lib.I8,
    torch.int16: _lib.I16,
    torch.int32: _lib.I32,
    torch.int64: _lib.I64,
    torch.float16: _lib.F16,
    torch.float32: _lib.F32,
    torch.float64: _lib.F64,
}


def _check(cond: bool, text: str) -> None:
    if not cond:
        raise RuntimeError(f"Check failed: {text}")


def _require_gpu(t: torch.Tensor) -> None:
    # visual_hull.cpp:70-82, marching_cubes.cpp:20-25, gaussian_blur.cpp:22-27
    if not t.is_cuda:
        raise RuntimeError(f'No backend implementation available for device "{t.device}".')


def _stream(device: torch.device) -> ctypes.c_void_p:
    return ctypes.c_void_p(torch.cuda.current_stream(device).cuda_stream)


def _ptr(t: torch.Tensor) -> ctypes.c_void_p:
    return ctypes.c_void_p(t.data_ptr())


def _convention(transforms_convention: str) -> int:
    if transforms_convention == "opengl":
        return 1
    if transforms_convention == "opencv":
        return 0
    raise RuntimeError(f'Unsupported transforms_convention "{transforms_convention}".')


def _masks_for_abi(masks: torch.Tensor) -> tuple[torch.Tensor, int]:
    """[B,H,W,1] masks -> contiguous [B,H,W] in a dtype the kernels read natively.

    float32, uint8 and bool are read as they are; every other dtype is converted
    to float32 first, which is what the reference does per sample
    (image_utils.h:178 casts to float) and for the integral (cumsum in float32)."""
    if masks.dtype in (torch.float32, torch.uint8, torch.bool) and masks.is_contiguous():
        return masks, _DTYPE_CODES[masks.dtype]  # [B,H,W,1] contiguous has the [B,H,W] layout
    m = masks[..., 0]
    if m.dtype in (torch.float32, torch.uint8, torch.bool):
        m = m.contiguous()
    else:
        m = m.to(torch.float32).contiguous()
    code = _DTYPE_CODES[m.dtype]
    return m, code


def _check_vh_args(masks: torch.Tensor, transforms: torch.Tensor, level: int, cube_length: float) -> torch.Size:
    """The argument checks of visual_hull.cpp:34-58; returns the masks' shape."""
    ms, ts = masks.shape, transforms.shape
    _check(masks.device == transforms.device, "masks.device() == transforms.device()")
    _check(len(ms) == 4, "masks.dim() == 4")
    _check(len(ts) == 3, "transforms.dim() == 3")
    _check(ts[1] == 4, "transforms.size(1) == 4")
    _check(ts[2] == 4, "transforms.size(2) == 4")
    _check(ms[0] == ts[0], "masks.size(0) == transforms.size(0)")
    _check(ms[3] == 1, "masks.size(3) == 1")
    _check(int(level) >= 0, "level >= 0")
    _check(float(cube_length) > 0.0, "cube_length > 0.f")
    return ms


_F3 = ctypes.c_float * 3


def _scene_struct(masks: torch.Tensor, transforms: torch.Tensor, level: int, cube_corner_bfl: Sequence[float],
                  cube_length: float, masks_partial: bool, transforms_convention: str,
                  keep: list) -> _lib.Scene:
    _require_gpu(masks)
    ms = _check_vh_args(masks, transforms, level, cube_length)
    opengl = _convention(transforms_convention)
    m, code = _masks_for_abi(masks)
    T = transforms
    if T.dtype != torch.float32 or not T.is_contiguous():
        T = T.to(torch.float32).contiguous()  # fmaf arguments are float (visual_hull_cuda.cu:150-153)
    keep.append(m)
    keep.append(T)
    c = cube_corner_bfl
    _check(len(c) == 3, "len(cube_corner_bfl) == 3")
    return _lib.Scene(m.data_ptr(), code, T.data_ptr(), ms[0], ms[1], ms[2], int(level), int(bool(masks_partial)),
                      opengl, _F3(float(c[0]), float(c[1]), float(c[2])), float(cube_length))


class _Run:
    """One visual-hull batch executed by the library; results stay in the context until the next call.

    join(step, last_step, room) -> list of _lib.Scene, if given, is asked at every level boundary for
    scenes that join the octree loop there (at most `room`, max_scenes in all); their results follow the
    initial scenes' in join order."""

    def __init__(self, scenes: list[_lib.Scene], device: torch.device, unique_verts: bool, join=None,
                 max_scenes: int | None = None) -> None:
        self.device = device
        self.ctx = _lib.context(device.index if device.index is not None else torch.cuda.current_device())
        self.stream = _stream(device)
        arr = (_lib.Scene * len(scenes))(*scenes)
        with torch.cuda.device(device):
            if join is None:
                self.counts = (_lib.VhCounts * len(scenes))()
                _lib.check(_lib.lib().thull_visual_hull_run(self.ctx, arr, len(scenes), int(bool(unique_verts)),
                                                            self.stream, self.counts))
                return
            cap = int(max_scenes if max_scenes is not None else len(scenes))
            counts = (_lib.VhCounts * cap)()
            failure: list = []

            def cb(_user, step, last_step, out, max_out):
                try:
                    new = list(join(int(step), int(last_step), int(max_out)))[:int(max_out)]
                    for k, sc in enumerate(new):
                        out[k] = sc
                    return len(new)
                except BaseException as e:  # noqa: BLE001 - re-raised after the run
                    failure.append(e)
                    return -1

            fn = _lib.JOIN_FN(cb)
            n_total = ctypes.c_int32()
            rc = _lib.lib().thull_visual_hull_run_join(self.ctx, arr, len(scenes), int(bool(unique_verts)),
                                                       self.stream, fn, None, cap, counts, ctypes.byref(n_total))
            if failure:
                raise failure[0]
            _lib.check(rc)
            self.counts = (_lib.VhCounts * n_total.value)(*counts[:n_total.value])

    def meshes(self) -> list[tuple[torch.Tensor, torch.Tensor]]:
        """All scenes' meshes with two copies: views into one vertex and one face tensor."""
        nv = [int(self.counts[i].num_verts) for i in range(len(self.counts))]
        nf = [int(self.counts[i].num_faces) for i in range(len(self.counts))]
        verts = torch.empty((sum(nv), 3), dtype=torch.float32, device=self.device)
        faces = torch.empty((sum(nf), 3), dtype=torch.int64, device=self.device)
        _lib.check(_lib.lib().thull_visual_hull_fetch_all(self.ctx, _ptr(verts), _ptr(faces), self.stream))
        out, v0, f0 = [], 0, 0
        for a, b in zip(nv, nf):
            out.append((verts[v0:v0 + a], faces[f0:f0 + b]))
            v0 += a
            f0 += b
        return out

    def mesh(self, i: int) -> tuple[torch.Tensor, torch.Tensor]:
        c = self.counts[i]
        verts = torch.empty((c.num_verts, 3), dtype=torch.float32, device=self.device)
        faces = torch.empty((c.num_faces, 3), dtype=torch.int64, device=self.device)
        _lib.check(_lib.lib().thull_visual_hull_fetch_mesh(self.ctx, i, _ptr(verts), _ptr(faces), self.stream))
        return verts, faces

    def field(self, i: int, level: int) -> torch.Tensor:
        c = self.counts[i]
        n = c.num_field
        idx = torch.empty((4, n), dtype=torch.int64, device=self.device)
        vals = torch.empty((n,), dtype=torch.float32, device=self.device)
        _lib.check(_lib.lib().thull_visual_hull_fetch_field(self.ctx, i, _ptr(idx), _ptr(vals), self.stream))
        r = (1 << level) + 1
        # to_sparse_coo_tensor (visual_hull_cuda.cu:575-577); indices are sorted and unique, so coalescing would
        # only sort them again (a level-8 field: 266 of 732 us) and add every value to zero, as here
        return torch.sparse_coo_tensor(idx, vals.add_(0.0), (1, r, r, r), is_coalesced=True)

    def candidates(self) -> list[torch.Tensor]:
        L = _lib.lib()
        out = []
        for level in range(self.counts[0].num_levels):
            n = ctypes.c_int64()
            _lib.check(L.thull_visual_hull_candidates_count(self.ctx, level, ctypes.byref(n)))
            t = torch.empty((n.value,), dtype=torch.int64, device=self.device)
            _lib.check(L.thull_visual_hull_fetch_candidates(self.ctx, level, _ptr(t), self.stream))
            out.append(t)
        return out


def visual_hull(masks: torch.Tensor, transforms: torch.Tensor, level: int, cube_corner_bfl: Sequence[float],
                cube_length: float, masks_partial: bool, transforms_convention: str,
                unique_verts: bool = True) -> tuple[torch.Tensor, torch.Tensor]:
    """Visual hull of the masks as a mesh (bindings.cpp:12-57, visual_hull.cpp:34-58).

    masks [B,H,W,1] (values in {0,1} or fractional), transforms [B,4,4]
    (intrinsics * extrinsics), cube [corner, corner + length]^3 at resolution
    2^level.  Returns verts float32 [V,3] and faces int64 [F,3]."""
    keep: list = []
    s = _scene_struct(masks, transforms, level, cube_corner_bfl, cube_length, masks_partial, transforms_convention,
                      keep)
    run = _Run([s], masks.device, unique_verts)
    return run.mesh(0)


def visual_hull_with_candidate_voxels(masks: torch.Tensor, transforms: torch.Tensor, level: int,
                                      cube_corner_bfl: Sequence[float], cube_length: float, masks_partial: bool,
                                      transforms_convention: str, unique_verts: bool = True
                                      ) -> tuple[torch.Tensor, torch.Tensor, list[torch.Tensor]]:
    """As visual_hull, plus the ravelled candidate cells of every level (bindings.cpp:59-105)."""
    keep: list = []
    s = _scene_struct(masks, transforms, level, cube_corner_bfl, cube_length, masks_partial, transforms_convention,
                      keep)
    run = _Run([s], masks.device, unique_verts)
    verts, faces = run.mesh(0)
    return verts, faces, run.candidates()


def sparse_visual_hull_field(masks: torch.Tensor, transforms: torch.Tensor, level: int,
                             cube_corner_bfl: Sequence[float], cube_length: float, masks_partial: bool,
                             transforms_convention: str) -> torch.Tensor:
    """Sparse field [1,R+1,R+1,R+1] (indices z, y, x) whose 0.5 isosurface is the hull (bindings.cpp:137-178)."""
    keep: list = []
    s = _scene_struct(masks, transforms, level, cube_corner_bfl, cube_length, masks_partial, transforms_convention,
                      keep)
    run = _Run([s], masks.device, True)
    return run.field(0, int(level))


def visual_hull_batch(scenes: Sequence[dict], unique_verts: bool = True,
                      graph: bool = False) -> list[tuple[torch.Tensor, torch.Tensor]]:
    """Visual hulls of many independent scenes in one batched pipeline run.

    Each scene is a dict with the keyword arguments of visual_hull (masks,
    transforms, level, cube_corner_bfl, cube_length, masks_partial,
    transforms_convention).  Every level of every scene is carved in one
    launch per octree level; results equal those of separate visual_hull calls.
    The meshes are views into one vertex tensor and one face tensor.

    graph=True: batches of a shape seen before (same scene count, cameras, image
    sizes, levels and flags) replay a captured hipGraph of the carving loop whose
    kernels read the level sizes on the device, with no host wait between levels
    (thull_ctx_set_graph_replay); the first batch of a shape is carved host-driven
    and leaves the plan.  Results are the same either way."""
    _check(len(scenes) > 0, "len(scenes) > 0")
    keep: list = []
    structs = []
    device = scenes[0]["masks"].device
    for sc in scenes:
        _check(sc["masks"].device == device, "all scenes on one device")
        structs.append(_scene_struct(sc["masks"], sc["transforms"], sc["level"], sc["cube_corner_bfl"],
                                     sc["cube_length"], sc["masks_partial"], sc["transforms_convention"], keep))
    if not graph:
        return _Run(structs, device, unique_verts).meshes()
    ctx = _lib.context(device.index if device.index is not None else torch.cuda.current_device())
    _lib.check(_lib.lib().thull_ctx_set_graph_replay(ctx, 1))
    try:
        run = _Run(structs, device, unique_verts)
    finally:
        _lib.check(_lib.lib().thull_ctx_set_graph_replay(ctx, 0))
    return run.meshes()


def graph_stats(device: torch.device | str | None = None) -> dict:
    """Carving-loop graphs captured, runs replayed from them and replays that overflowed their plan, on the
    calling thread's context of `device`."""
    dev = torch.device(device) if device is not None else torch.device("cuda", torch.cuda.current_device())
    ctx = _lib.context(dev.index if dev.index is not None else torch.cuda.current_device())
    c, r, o = ctypes.c_int64(), ctypes.c_int64(), ctypes.c_int64()
    _lib.check(_lib.lib().thull_ctx_graph_stats(ctx, ctypes.byref(c), ctypes.byref(r), ctypes.byref(o)))
    return {"captures": c.value, "replays": r.value, "overflows": o.value}


def candidate_voxels_to_wireframes(candidate_voxels: Sequence[torch.Tensor], cube_corner_bfl: Sequence[float],
                                   cube_length: float) -> list[tuple[torch.Tensor, torch.Tensor]]:
    """Wireframes of the candidate cells of every level (bindings.cpp:107-135, visual_hull_cuda.cu:1022-1111).

    Level i cells are ravelled at resolution 2^i; each cell gives 8 vertices
    fmaf(length / 2^i, corner_index, cube_corner) (float32 [8N,3]) and 12 edges (int64 [12N,2])."""
    _check(len(candidate_voxels) > 0, "candidate_voxels.empty() == false")
    for c in candidate_voxels:
        _check(c.device == candidate_voxels[0].device, "candidates.device() == candidate_voxels[0].device()")
    _require_gpu(candidate_voxels[0])
    device = candidate_voxels[0].device
    _check(len(cube_corner_bfl) == 3, "len(cube_corner_bfl) == 3")
    corner = _F3(*(float(v) for v in cube_corner_bfl))
    ctx = _lib.context(device.index if device.index is not None else torch.cuda.current_device())
    st = _stream(device)
    out = []
    with torch.cuda.device(device):
        for i, cand in enumerate(candidate_voxels):
            _check(cand.dtype == torch.int64, "candidates.dtype() == torch::kInt64")
            c = cand.reshape(-1).contiguous()
            n = c.numel()
            verts = torch.empty((8 * n, 3), dtype=torch.float32, device=device)
            edges = torch.empty((12 * n, 2), dtype=torch.int64, device=device)
            _lib.check(_lib.lib().thull_candidate_wireframe(ctx, _ptr(c), n, i, corner, float(cube_length),
                                                            _ptr(verts), _ptr(edges), st))
            out.append((verts, edges))
    return out


def marching_cubes(volume: torch.Tensor, isolevel: float, return_local_coords: bool = True,
                   unique_verts: bool = True) -> tuple[torch.Tensor, torch.Tensor]:
    """Marching cubes on a dense [1,D,H,W] or sparse COO volume (bindings.cpp:180-214, marching_cubes_cuda.cu:817-831)."""
    _require_gpu(volume)
    _check(volume.size(0) == 1, "volume.size(0) == 1")
    _check(float(isolevel) >= 0, "isolevel >= 0")
    device = volume.device
    ctx = _lib.context(device.index if device.index is not None else torch.cuda.current_device())
    st = _stream(device)
    L = _lib.lib()
    nv, nf = ctypes.c_int64(), ctypes.c_int64()
    with torch.cuda.device(device):
        if volume.is_sparse:
            _check(volume.sparse_dim() == 4, "volume.sparse_dim() == 4")
            _check(volume.dense_dim() == 0, "volume.dense_dim() == 0")
            _check(volume.values().numel() < (1 << 31), "volume.values().numel() < 2^31")
            v = volume if volume.is_coalesced() else volume.coalesce()
            idx = v.indices().contiguous()
            vals = v.values()
            if vals.dtype not in (torch.float32, torch.float64):
                vals = vals.to(torch.float32)
            vals = vals.contiguous()
            D, H, W = (int(s) for s in volume.shape[1:])
            # indices outside the volume are found, and refused, by the library as it reads them
            _check(vals.numel() == 0 or min(D, H, W) > 0, "indices within the volume")
            _lib.check(L.thull_marching_cubes_sparse_run(ctx, _ptr(idx), _ptr(vals), _DTYPE_CODES[vals.dtype],
                                                         vals.numel(), D, H, W, float(isolevel),
                                                         int(bool(return_local_coords)), int(bool(unique_verts)), st,
                                                         ctypes.byref(nv), ctypes.byref(nf)))
        else:
            _check(volume.dim() == 4, "volume.dim() == 4")
            vol = volume if volume.dtype in (torch.float32, torch.float64) else volume.to(torch.float32)
            vol = vol.contiguous()
            D, H, W = (int(s) for s in volume.shape[1:])
            _lib.check(L.thull_marching_cubes_dense_run(ctx, _ptr(vol), _DTYPE_CODES[vol.dtype], D, H, W,
                                                        float(isolevel), int(bool(return_local_coords)),
                                                        int(bool(unique_verts)), st, ctypes.byref(nv),
                                                        ctypes.byref(nf)))
        verts = torch.empty((nv.value, 3), dtype=torch.float32, device=device)
        faces = torch.empty((nf.value, 3), dtype=torch.int64, device=device)
        _lib.check(L.thull_marching_cubes_fetch(ctx, _ptr(verts), _ptr(faces), st))
    return verts, faces


def gaussian_blur(images: torch.Tensor, kernel_size: int, sigma: float, sparse: bool = True,
                  dtype: torch.dtype | None = None) -> torch.Tensor:
    """Gaussian blur of [B,H,W,C] images (bindings.cpp:216-251); the band blur (sparse=True) touches only
    pixels near mask edges of channel 0, every other value is the input converted to `dtype`."""
    _require_gpu(images)
    _check(int(kernel_size) > 0, "kernel_size > 0")
    _check(int(kernel_size) % 2 == 1, "kernel_size % 2 == 1")
    _check(float(sigma) > 0.0, "sigma > 0.f")
    _check(images.dim() == 4, "images.dim() == 4")
    out_dtype = images.dtype if dtype is None else dtype
    _check(out_dtype in (torch.float16, torch.float32, torch.float64), "isFloatingType(dtype)")
    if images.dtype not in _DTYPE_CODES:
        raise RuntimeError(f"gaussian_blur: unsupported input dtype {images.dtype}")
    device = images.device
    B, H, W, C = (int(s) for s in images.shape)
    src = images[..., 0].contiguous()
    ctx = _lib.context(device.index if device.index is not None else torch.cuda.current_device())
    st = _stream(device)
    with torch.cuda.device(device):
        out0 = torch.empty((B, H, W), dtype=out_dtype, device=device)
        _lib.check(_lib.lib().thull_gaussian_blur(ctx, _ptr(src), _DTYPE_CODES[images.dtype], B, H, W,
                                                  int(kernel_size), float(sigma), int(bool(sparse)), _ptr(out0),
                                                  _DTYPE_CODES[out_dtype], st))
        if C == 1:
            return out0.unsqueeze(-1)
        if not sparse and int(kernel_size) > 1:
            # the dense reference convolves every channel with the same kernel (gaussian_blur_cuda.cu:94-109)
            chans = [out0]
            for c in range(1, C):
                sc = images[..., c].contiguous()
                oc = torch.empty((B, H, W), dtype=out_dtype, device=device)
                _lib.check(_lib.lib().thull_gaussian_blur(ctx, _ptr(sc), _DTYPE_CODES[images.dtype], B, H, W,
                                                          int(kernel_size), float(sigma), 0, _ptr(oc),
                                                          _DTYPE_CODES[out_dtype], st))
                chans.append(oc)
            return torch.stack(chans, dim=-1)
        # sparse: only channel 0 is blurred (gaussian_blur_cuda.cu:221,230); the rest is the converted input
        out = images.to(out_dtype).clone()
        out[..., 0] = out0
        return out


def gaussian_blur_batch(images: Sequence[torch.Tensor], kernel_size: int, sigma: float, sparse: bool = True,
                        dtype: torch.dtype | None = None, context=None) -> list[torch.Tensor]:
    """gaussian_blur of many [B,H,W,1] tensors (one input dtype, one device) in one launch per pass.

    Each result equals gaussian_blur(images[i], kernel_size, sigma, sparse, dtype).  `context`: a library
    context other than the thread's own (the request server blurs joining scenes while its context runs)."""
    _check(len(images) > 0, "len(images) > 0")
    device = images[0].device
    _require_gpu(images[0])
    _check(int(kernel_size) > 0, "kernel_size > 0")
    _check(int(kernel_size) % 2 == 1, "kernel_size % 2 == 1")
    _check(float(sigma) > 0.0, "sigma > 0.f")
    in_dtype = images[0].dtype
    out_dtype = in_dtype if dtype is None else dtype
    _check(out_dtype in (torch.float16, torch.float32, torch.float64), "isFloatingType(dtype)")
    if in_dtype not in _DTYPE_CODES:
        raise RuntimeError(f"gaussian_blur: unsupported input dtype {in_dtype}")
    srcs, outs, sizes = [], [], []
    for im in images:
        _check(im.device == device and im.dtype == in_dtype, "one device and dtype per batch")
        _check(im.dim() == 4 and im.size(3) == 1, "images [B,H,W,1]")
        srcs.append(im if im.is_contiguous() else im[..., 0].contiguous())  # [B,H,W,1] contiguous = [B,H,W]
        outs.append(torch.empty(tuple(im.shape), dtype=out_dtype, device=device))
        sizes.extend(int(v) for v in im.shape[:3])
    n = len(images)
    src_p = (ctypes.c_void_p * n)(*[t.data_ptr() for t in srcs])
    out_p = (ctypes.c_void_p * n)(*[t.data_ptr() for t in outs])
    sz = (ctypes.c_int64 * (3 * n))(*sizes)
    ctx = context if context is not None else _lib.context(
        device.index if device.index is not None else torch.cuda.current_device())
    with torch.cuda.device(device):
        _lib.check(_lib.lib().thull_gaussian_blur_batch(ctx, n, src_p, _DTYPE_CODES[in_dtype], sz, int(kernel_size),
                                                        float(sigma), int(bool(sparse)), out_p,
                                                        _DTYPE_CODES[out_dtype], _stream(device)))
    return outs


def _format_float_like_ostream(x: float) -> str:
    """A float as std::ostream << float writes it by default (printf %g, precision 6; glibc spells a
    NaN with the sign bit set "-nan")."""
    if math.isnan(x):
        return "-nan" if math.copysign(1.0, x) < 0 else "nan"
    return f"{x:g}"


def store_curve_network(filename: str, curve_network: tuple[torch.Tensor, torch.Tensor],
                        verbose: bool = False) -> None:
    """Writes a curve network (vertices [V,3], edges [E,2]) as OBJ text (1-indexed `l` lines) or as
    binary little-endian PLY with float32 vertices and int32 edges, chosen by the extension (io.cpp:11-127)."""
    path = pathlib.Path(filename)
    suffix = path.suffix
    if suffix not in (".obj", ".ply"):
        raise RuntimeError(f'No implementation for file extension "{suffix}".')
    if verbose:
        print(f'Storing file "{filename}" ...', flush=True)
    t0 = time.perf_counter()
    verts, edges = curve_network
    v = verts.detach().to("cpu", torch.float32).contiguous()
    e = edges.detach().to("cpu", torch.int64).contiguous()
    if suffix == ".obj":
        with open(path, "w") as f:
            for x, y, z in v.tolist():
                f.write(f"v {_format_float_like_ostream(x)} {_format_float_like_ostream(y)} "
                        f"{_format_float_like_ostream(z)}\n")
            for a, b in e[:, :2].tolist():
                f.write(f"l {a + 1} {b + 1}\n")  # 1-indexed
    else:
        import numpy as np

        header = ("ply\nformat binary_little_endian 1.0\n"
                  f"element vertex {v.shape[0]}\nproperty float x\nproperty float y\nproperty float z\n"
                  f"element edge {e.shape[0]}\nproperty int vertex1\nproperty int vertex2\nend_header\n")
        with open(path, "wb") as f:
            f.write(header.encode("ascii"))
            f.write(np.ascontiguousarray(v.numpy(), dtype="<f4").tobytes())
            # edges as int32 (torch's int64 -> int32 conversion keeps the low 32 bits)
            f.write(np.ascontiguousarray(e.numpy().astype(np.int32), dtype="<i4").tobytes())
    if verbose:
        ms = int((time.perf_counter() - t0) * 1000)
        print(f'Storing file "{filename}" ... done ({ms / 1000:g}s)', flush=True)
