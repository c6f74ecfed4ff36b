"""Corner vertices numbered by groups of words that kept bricks reach: hulls that touch the grid's far and near borders,
where the last word of a row, the last rows and the last planes hold vertices."""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch

from tests.gpu_util import DEV
from tests.test_gpu_solid_maps import _check
from torchhull_amd import synthetic

pytestmark = pytest.mark.gpu


def _border_scene(cameras, size, sign):
    rng = np.random.default_rng(31)
    centers = sign * np.array([[0.8, 0.75, 0.7], [0.1, 0.9, -0.2], [0.85, -0.1, 0.3]])  # out of the cube [-1, 1]^3
    axes = rng.uniform(0.25, 0.45, size=(3, 3))
    rot = np.stack([synthetic.random_rotation(rng) for _ in range(3)])
    fovy = math.radians(50.0)
    views = np.stack([synthetic.look_at(e) for e in synthetic.fibonacci_cameras(cameras, 3.5)])
    masks = synthetic.render_masks_gl(views, fovy, size, size, centers, rot, axes)
    T = np.einsum("ij,bjk->bik", synthetic.perspective(fovy, 1.0, 0.1, 1000.0), views)
    return masks.contiguous().numpy(), T.astype(np.float32)


@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("cameras, size, level", [(36, 230, 9), (9, 310, 10)])
def test_hull_at_the_border(cameras, size, level, sign):
    masks, T = _border_scene(cameras, size, sign)
    print(f"case border level={level} sign={sign}", flush=True)
    assert _check(masks, T, level, False, "opengl") > 0


def test_tiles_of_several_scenes_equal_single_calls():
    # 4096 words of a numbering tile hold many scenes of levels 0 to 4 beside one that takes the batch to bricks
    import torchhull_amd as th

    scenes = []
    for i, level in enumerate((4, 0, 3, 9, 1, 2, 4, 4, 0, 3, 3, 2)):
        masks, T = _border_scene(40 if level == 9 else 4, 200, 1.0 if i % 2 else -1.0)
        scenes.append(dict(masks=torch.from_numpy(masks).to(DEV), transforms=torch.from_numpy(T).to(DEV), level=level,
                           cube_corner_bfl=(-1.0, -1.0, -1.0), cube_length=2.0, masks_partial=False,
                           transforms_convention="opengl"))
    print("case several scenes per tile", flush=True)
    for s, (v, f) in zip(scenes, th.visual_hull_batch(scenes)):
        va, fa = th.visual_hull(**s)
        assert torch.equal(fa, f) and torch.equal(va.view(torch.int32), v.view(torch.int32))


def test_scenes_that_join_a_loop_by_bricks_equal_single_calls():
    # scenes handed over at level boundaries of a loop that keeps bricks: their descriptors, maps, bitmaps and flags
    # are added while the loop runs
    import torchhull_amd as th
    from torchhull_amd import api

    scenes = []
    for i, (cameras, level) in enumerate(((40, 9), (12, 6), (36, 7), (5, 0), (6, 4))):
        masks, T = _border_scene(cameras, 200, 1.0 if i % 2 else -1.0)
        scenes.append(dict(masks=torch.from_numpy(masks).to(DEV), transforms=torch.from_numpy(T).to(DEV), level=level,
                           cube_corner_bfl=(-1.0, -1.0, -1.0), cube_length=2.0, masks_partial=False,
                           transforms_convention="opengl"))
    keep: list = []
    structs = [api._scene_struct(**s, keep=keep) for s in scenes]
    steps = {2: [structs[1], structs[2]], 5: [structs[3], structs[4]]}
    print("case joining scenes", flush=True)
    run = api._Run(structs[:1], torch.device(DEV), True, join=lambda step, last, room: steps.pop(step, []),
                   max_scenes=len(structs))
    meshes = run.meshes()
    assert len(meshes) == len(scenes)
    for s, (v, f) in zip(scenes, meshes):
        va, fa = th.visual_hull(**s)
        assert torch.equal(fa, f) and torch.equal(va.view(torch.int32), v.view(torch.int32))
