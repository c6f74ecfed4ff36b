"""The carving kernel that the profile names for each step is the one that ran (thull_profile_carve)."""

from __future__ import annotations

import concurrent.futures
import ctypes

import pytest
import torch

from tests.gpu_util import DEV
from tests.test_gpu_solid_maps import CORNER, LENGTH, _scene

pytestmark = pytest.mark.gpu


def _profile(run):
    from torchhull_amd import _lib

    ctx, L, n = _lib.context(0), _lib.lib(), 16
    _lib.check(L.thull_profile_enable(ctx, 1))
    try:
        run()
    finally:
        _lib.check(L.thull_profile_enable(ctx, 0))
    ms, split = (ctypes.c_float * n)(), (ctypes.c_int32 * n)()
    parents, tests, children = ((ctypes.c_int64 * n)() for _ in range(3))
    _lib.check(L.thull_profile_carve(ctx, n, ms, parents, tests, children, split))
    return [(int(p), int(s)) for p, s in zip(parents, split) if p > 0]


def _expected(parents, cameras, max_parents):
    """kChildSplit up to 8192 wavefronts of 64-lane levels, then the thresholds' lanes as far as cameras fill them."""
    lanes = next((g for g, most in zip((64, 16, 4, 2), max_parents) if parents <= most), 1)
    group = max(8, 1 << (cameras - 1).bit_length())
    if lanes == 64 and parents * group // 8 <= 8192:
        return 8
    if lanes == 64 and cameras <= 16:
        lanes = 16
    return 4 if lanes == 16 and cameras <= 4 else lanes


def _check(cameras):
    import torchhull_amd as th
    from torchhull_amd import _lib, tuning

    tuning.set_carve_tuning(_lib.context(0), (30000, 50000, 60000, 100000))
    masks, T = _scene(51, cameras, 160, 150, "opengl")
    scene = dict(masks=torch.from_numpy(masks).to(DEV), transforms=torch.from_numpy(T).to(DEV), level=8,
                 cube_corner_bfl=CORNER, cube_length=LENGTH, masks_partial=False, transforms_convention="opengl")
    print(f"case {cameras} cameras", flush=True)
    driven = _profile(lambda: th.visual_hull(**scene))
    assert [s for _, s in driven] == [_expected(p, cameras, (30000, 50000, 60000, 100000)) for p, _ in driven]
    assert 8 in [s for _, s in driven]
    th.visual_hull_batch([scene], graph=True)  # leaves the plan: levels at a quarter more than their size
    replayed = _profile(lambda: th.visual_hull_batch([scene], graph=True))
    assert [p for p, _ in replayed] == [p for p, _ in driven]
    for (parents, a), (_, b) in zip(driven, replayed):
        assert b == {1: 0}.get(a, a) or a == 8  # a level of the smallest kernel may round up out of its range


@pytest.mark.parametrize("cameras", [3, 12, 20, 40])
def test_the_profile_names_the_kernels(cameras):
    with concurrent.futures.ThreadPoolExecutor(1) as pool:  # a context of its own: its tuning ends with it
        pool.submit(_check, cameras).result()
