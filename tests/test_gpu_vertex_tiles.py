"""Numbering of the corner vertices on small and on large bitmaps (up to and beyond 2^23 words) without brick lists."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle
from tests.gpu_util import DEV, assert_mesh_equal
from tests.test_gpu_solid_maps import CORNER, LENGTH, _scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level", [1, 2, 4, 5, 6, 9, 10])
def test_vertices_of_bitmaps(level):
    import torchhull_amd as th

    masks, T = _scene(81, 5, 180, 200, "opengl")
    assert T.shape[0] << (2 * level) < 1 << 23  # no brick lists
    args = (torch.from_numpy(masks).to(DEV), torch.from_numpy(T).to(DEV), level, CORNER, LENGTH, False, "opengl")
    print(f"case bitmap level={level}", flush=True)
    field = th.sparse_visual_hull_field(*args)
    fld = oracle.sparse_field(masks, T, level, CORNER, LENGTH, False, "opengl")
    assert np.array_equal(field.values().cpu().numpy().view(np.uint32), fld.values.view(np.uint32))
    v, f = th.visual_hull(*args)
    ov, of = oracle.visual_hull(None, None, level, CORNER, LENGTH, False, "opengl", True, field=fld)
    assert_mesh_equal(v, f, ov, of, atol=1e-6 * LENGTH)


def test_vertices_of_a_batch_of_small_bitmaps():
    # tiles of 512 words that hold several scenes
    import torchhull_amd as th

    scenes = []
    for i, level in enumerate((3, 0, 1, 5, 2, 0, 4, 1, 6, 3)):
        masks, T = _scene(90 + i, 4, 64, 64, "opengl")
        scenes.append(dict(masks=torch.from_numpy(masks).to(DEV), transforms=torch.from_numpy(T).to(DEV), level=level,
                           cube_corner_bfl=CORNER, cube_length=LENGTH, masks_partial=False,
                           transforms_convention="opengl"))
    print("case batch of small bitmaps", flush=True)
    for s, (v, f) in zip(scenes, th.visual_hull_batch(scenes)):
        va, fa = th.visual_hull(**s)
        assert torch.equal(f, fa) and torch.equal(v, va)
