"""Octree levels around the largest one that is compacted in one launch (2^17 parents): half-tone masks keep every cell,
so that batches of n level-6 scenes have n * 2^15 parents at their last step."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle
from tests.gpu_util import DEV
from tests.test_gpu_solid_maps import CORNER, LENGTH, _scene

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
