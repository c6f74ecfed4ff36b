"""Dense marching cubes at the edges of its words, tiles and queues: row lengths around whole 32-point words, row
counts around the sign pass's groups of 4, volumes around one and several tiles of 256 words, and volumes in
which (nearly) every cell has triangles."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle
from tests.gpu_util import DEV, assert_mesh_equal

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 2), (2, 2, 31), (2, 3, 32), (3, 2, 33), (5, 7, 63), (2, 5, 64), (3, 3, 65), (2, 512, 32),
          (2, 513, 31), (4, 256, 40), (5, 205, 30), (3, 171, 97), (40, 2, 2), (2, 1030, 3)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("unique_verts", [True, False])
def test_dense_words_and_tiles_match_oracle(shape, dtype, unique_verts):
    import torchhull_amd as th

    rng = np.random.default_rng(sum(shape) + 7 * shape[2])
    vol = rng.uniform(-1, 1, size=shape).astype(dtype)
    vol[:, : shape[1] // 3] = np.abs(vol[:, : shape[1] // 3]) + 1.0  # a part without surface
    if shape[1] > 4:
        vol[0, -1, -1] = np.nan  # compares as not below the isolevel
    print(f"case {shape} {dtype.__name__} unique={unique_verts}", flush=True)
    v, f = th.marching_cubes(torch.from_numpy(vol)[None].to(DEV), 0.25, return_local_coords=False,
                             unique_verts=unique_verts)
    ov, of = oracle.marching_cubes_dense(vol, 0.25, unique_verts)
    assert_mesh_equal(v, f, ov, of, atol=1e-6 * max(shape))
