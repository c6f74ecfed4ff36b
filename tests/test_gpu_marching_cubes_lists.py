"""Sparse marching cubes at the edges of its entry marking: rows that end inside, at and past a 32-bit bitmap
word, lists that end inside a wavefront, and indices that must be refused."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle
from tests.gpu_util import DEV, assert_mesh_equal

pytestmark = pytest.mark.gpu


def _th():
    import torchhull_amd as th

    return th


@pytest.mark.parametrize("width", [2, 31, 32, 33, 63, 64, 65, 97])
@pytest.mark.parametrize("density", [0.97, 0.6])
def test_sparse_rows_across_bitmap_words_match_oracle(width, density):
    th = _th()
    rng = np.random.default_rng(width * 100 + int(10 * density))
    D, H, W = 5, 7, width
    vol = rng.normal(size=(D, H, W)).astype(np.float32)
    keep = rng.uniform(size=(D, H, W)) < density
    keep[2:4, 2:4, :2] = True  # at least one complete cell
    z, y, x = np.nonzero(keep)
    idx = torch.from_numpy(np.stack([np.zeros_like(z), z, y, x]))
    vals = vol[z, y, x]
    sp = torch.sparse_coo_tensor(idx, torch.from_numpy(vals), (1, D, H, W)).coalesce()
    print(f"case {D}x{H}x{W} nnz {len(vals)}", flush=True)
    v, f = th.marching_cubes(sp.to(DEV), 0.25, return_local_coords=False)
    ids = x + W * (y + H * z)
    ov, of = oracle.marching_cubes_sparse(ids, vals, (W, H, D), 0.25, True)
    assert_mesh_equal(v, f, ov, of, atol=1e-6 * max(D, H, W))


@pytest.mark.parametrize("row,value", [(0, -1), (1, 4), (2, 4), (3, 4), (1, -1), (2, -1), (3, -1)])
@pytest.mark.parametrize("count", [1, 100])
def test_sparse_indices_outside_the_volume_are_refused(row, value, count):
    th = _th()
    idx = torch.zeros((4, count), dtype=torch.int64)
    at = torch.arange(count)
    idx[1], idx[2], idx[3] = (at // 16) % 4, (at // 4) % 4, at % 4
    idx[row, -1] = value
    sp = torch.sparse_coo_tensor(idx.to(DEV), torch.ones(count, device=DEV), (1, 4, 4, 4), is_coalesced=True)
    with pytest.raises(RuntimeError, match="indices within the volume"):
        th.marching_cubes(sp, 0.5)


def test_repeated_sparse_indices_of_a_tensor_marked_coalesced_are_refused():
    th = _th()
    idx = torch.zeros((4, 70), dtype=torch.int64)  # one entry 70 times: runs of equal words longer than a wave
    sp = torch.sparse_coo_tensor(idx.to(DEV), torch.ones(70, device=DEV), (1, 4, 4, 4), is_coalesced=True)
    with pytest.raises(RuntimeError, match="coalesced"):
        th.marching_cubes(sp, 0.5)
