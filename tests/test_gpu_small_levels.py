"""Small octree levels: around the largest one that is compacted in one launch (2^17 parents; half-tone masks keep every
cell, so that batches of n level-6 scenes have n * 2^15 parents at their last step), and the camera counts, conventions
and scene mixtures of the kernel for the smallest ones."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from oracle import oracle
from tests.gpu_util import DEV
from tests.test_gpu_solid_maps import CORNER, LENGTH, _scene
from torchhull_amd import _lib

pytestmark = pytest.mark.gpu


def _scene_dict(masks, T, level):
    return dict(masks=torch.from_numpy(masks).to(DEV), transforms=torch.from_numpy(T).to(DEV), level=level,
                cube_corner_bfl=CORNER, cube_length=LENGTH, masks_partial=False, transforms_convention="opengl")


@pytest.mark.parametrize("scenes", [1, 3, 4, 5])
def test_full_levels(scenes):
    import torchhull_amd as th

    masks, T = _scene(41, 2, 40, 40, "opengl")
    masks = np.full_like(masks, 0.5)
    fld = oracle.sparse_field(masks, T, 6, CORNER, LENGTH, False, "opengl")
    assert len(fld.candidates[5]) == 1 << 15
    s = _scene_dict(masks, T, 6)
    print(f"case full levels scenes={scenes}", flush=True)
    _, _, cand = th.visual_hull_with_candidate_voxels(**s)
    for a, b in zip(cand, fld.candidates):
        assert np.array_equal(a.cpu().numpy(), b)
    # half of the masks' height empty: other counts per block beside the full ones
    cut = masks.copy()
    cut[:, :17] = 0.0
    batch = [s] * (scenes - 1) + [_scene_dict(cut, T, 6)]
    singles = [th.visual_hull(**b) for b in (s, batch[-1])]
    for i, (v, f) in enumerate(th.visual_hull_batch(batch)):
        va, fa = singles[1 if i == scenes - 1 else 0]
        assert torch.equal(f, fa) and torch.equal(v, va)


@pytest.mark.parametrize("convention", ["opengl", "opencv"])
@pytest.mark.parametrize("partial", [False, True])
@pytest.mark.parametrize("cameras", [1, 4, 5, 8, 9, 16, 17, 33, 64, 65, 130])
def test_camera_counts_of_the_smallest_levels(cameras, partial, convention):
    # a lane per parent, child and camera: groups of 8 to 64 lanes, one or several rounds, levels within and beyond
    # the number of parents it is used for
    import torchhull_amd as th

    masks, T = _scene(50 + cameras, cameras, 61, 77, convention)
    args = (torch.from_numpy(masks).to(DEV), torch.from_numpy(T).to(DEV), 7, CORNER, LENGTH, partial, convention)
    print(f"case cameras={cameras} partial={partial} {convention}", flush=True)
    _, _, cand = th.visual_hull_with_candidate_voxels(*args)
    tests = (ctypes.c_int64 * 16)()
    _lib.check(_lib.lib().thull_visual_hull_stats(_lib.context(0), 16, tests, None))
    fld = oracle.sparse_field(masks, T, 7, CORNER, LENGTH, partial, convention)
    assert len(cand) == len(fld.candidates)
    for a, b in zip(cand, fld.candidates):
        assert np.array_equal(a.cpu().numpy(), b)
    assert list(tests)[:len(fld.tests)] == list(fld.tests)


def test_smallest_levels_of_a_mixed_batch():
    # parents of several scenes in one wavefront, with different conventions, partial flags and levels
    import torchhull_amd as th

    scenes = []
    for i, (cameras, level, partial, convention) in enumerate(((3, 5, False, "opengl"), (20, 6, True, "opencv"),
                                                               (8, 0, False, "opengl"), (7, 4, True, "opengl"),
                                                               (12, 6, False, "opencv"), (5, 1, True, "opencv"))):
        masks, T = _scene(70 + i, cameras, 50 + i, 64, convention)
        scenes.append(dict(masks=torch.from_numpy(masks).to(DEV), transforms=torch.from_numpy(T).to(DEV), level=level,
                           cube_corner_bfl=CORNER, cube_length=LENGTH, masks_partial=partial,
                           transforms_convention=convention))
    print("case mixed batch", flush=True)
    for s, (v, f) in zip(scenes, th.visual_hull_batch(scenes)):
        va, fa = th.visual_hull(**s)
        assert torch.equal(f, fa) and torch.equal(v, va)
