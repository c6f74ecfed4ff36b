"""Hulls large enough for solid maps (cameras left out of cells whose surroundings their masks fill) against the
oracle: every level's candidates, the canonical camera-test counts, field values bit for bit and the mesh."""

from __future__ import annotations

import ctypes
import math

import numpy as np
import pytest
import torch

from oracle import oracle
from tests.gpu_util import DEV, assert_mesh_equal
from torchhull_amd import synthetic

pytestmark = pytest.mark.gpu

CORNER, LENGTH = (-1.0, -1.0, -1.0), 2.0


def _scene(seed, cameras, height, width, convention, radius=2.5, fovy_deg=40.0):
    rng = np.random.default_rng(seed)
    n = 4
    centers = rng.uniform(-0.35, 0.35, size=(n, 3))
    axes = rng.uniform(0.2, 0.45, size=(n, 3))
    rot = np.stack([synthetic.random_rotation(rng) for _ in range(n)])
    fovy = math.radians(fovy_deg)
    views = np.stack([synthetic.look_at(e) for e in synthetic.fibonacci_cameras(cameras, radius)])
    masks = synthetic.render_masks_gl(views, fovy, height, width, centers, rot, axes)
    if convention == "opengl":
        T = np.einsum("ij,bjk->bik", synthetic.perspective(fovy, width / height, 0.1, 1000.0), views)
    else:
        D = np.diag([1.0, -1.0, -1.0, 1.0])
        T = np.einsum("ij,bjk->bik", synthetic.perspective_cv(fovy, width / height, height, width),
                      np.einsum("ij,bjk,kl->bil", D, views, D))
        masks = masks.flip(1)
    return masks.contiguous().numpy(), T.astype(np.float32)


def _check(masks, T, level, partial, convention):
    import torchhull_amd as th
    from torchhull_amd import _lib

    assert T.shape[0] << (2 * level) >= 1 << 23  # the maps are in use
    args = (torch.from_numpy(masks).to(DEV), torch.from_numpy(T).to(DEV), level, CORNER, LENGTH, partial, convention)
    v, f, cand = th.visual_hull_with_candidate_voxels(*args)
    tests = (ctypes.c_int64 * 16)()
    _lib.check(_lib.lib().thull_visual_hull_stats(_lib.context(0), 16, tests, None))
    field = th.sparse_visual_hull_field(*args)
    fld = oracle.sparse_field(masks, T, level, CORNER, LENGTH, partial, convention)
    for i, (a, b) in enumerate(zip(cand, fld.candidates)):
        assert np.array_equal(a.cpu().numpy(), b), f"candidates of level {i}"
    assert list(tests)[:len(fld.tests)] == list(fld.tests)
    assert np.array_equal(field.values().cpu().numpy().view(np.uint32), fld.values.view(np.uint32))
    ov, of = oracle.visual_hull(None, None, level, CORNER, LENGTH, partial, convention, True, field=fld)
    assert_mesh_equal(v, f, ov, of, atol=1e-6 * LENGTH)
    return f.shape[0]


@pytest.mark.parametrize("convention", ["opengl", "opencv"])
@pytest.mark.parametrize("partial", [False, True])
@pytest.mark.parametrize("dtype", [np.float32, np.uint8])
def test_binary_masks_of_odd_sizes(convention, partial, dtype):
    masks, T = _scene(11, 33, 331, 450, convention, *((1.6, 60.0) if partial else ()))
    print(f"case binary {convention} partial={partial} {dtype.__name__}", flush=True)
    assert _check(masks.astype(dtype), T, 9, partial, convention) > 1000


@pytest.mark.parametrize("kind", ["blurred", "nan", "negative", "large", "plateau", "255"])
def test_masks_that_limit_the_maps(kind):
    masks, T = _scene(12, 36, 320, 322, "opengl")
    if kind == "blurred":
        masks = oracle.gaussian_blur_sparse(masks, 7, 1.5, np.float32)
    elif kind == "nan":
        masks[::5, 200, 3] = np.nan
    elif kind == "negative":
        masks[::4, 3:9, 3:9] = -0.25
    elif kind == "large":
        masks[::3] *= 3.0
    elif kind == "plateau":
        masks[::2] *= np.float32(0.9990234375)
    else:
        masks = (masks * 255).astype(np.uint8)
    print(f"case {kind}", flush=True)
    _check(masks, T, 9, kind == "negative", "opengl")


def test_more_cameras_than_one_mask_word():
    masks, T = _scene(13, 70, 200, 260, "opencv")
    print("case 70 cameras", flush=True)
    assert _check(masks, T, 9, False, "opencv") > 1000


def test_more_cameras_than_the_brick_masks_hold():
    masks, T = _scene(14, 1100, 64, 80, "opengl")
    print("case 1100 cameras", flush=True)
    assert _check(masks, T, 7, False, "opengl") > 100


@pytest.mark.parametrize("partial", [False, True])
def test_cameras_among_the_cells(partial):
    # cameras inside the cube: denominators cross zero within cells
    masks, T = _scene(15, 34, 240, 240, "opengl", 0.6, 90.0)
    print(f"case cameras inside the cube partial={partial}", flush=True)
    _check(masks, T, 9, partial, "opengl")


def test_batch_of_scenes_with_and_without_maps_equals_single_calls():
    import torchhull_amd as th

    scenes = []
    for seed, cams, size, level, partial in ((21, 40, 300, 9, False), (22, 2, 120, 6, False), (23, 12, 14, 5, True),
                                             (24, 9, 260, 2, False), (25, 7, 200, 8, True), (26, 5, 90, 0, False),
                                             (27, 6, 150, 1, False)):
        masks, T = _scene(seed, cams, size, size, "opengl")
        scenes.append(dict(masks=torch.from_numpy(masks).to(DEV), transforms=torch.from_numpy(T).to(DEV), level=level,
                           cube_corner_bfl=CORNER, cube_length=LENGTH, masks_partial=partial,
                           transforms_convention="opengl"))
    print("case mixed batch", flush=True)
    for s, (v, f) in zip(scenes, th.visual_hull_batch(scenes)):
        va, fa = th.visual_hull(**s)
        assert torch.equal(fa, f) and torch.equal(va.view(torch.int32), v.view(torch.int32))
