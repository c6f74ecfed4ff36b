"""Carving that leaves out cameras under every launch shape that has code for it (4, 2 and 1 lanes per parent, and
the work-queue kernel of replayed carving loops), for partial masks, both conventions and more than 64 cameras: each
against the oracle or the host-driven loop, with the canonical camera-test counts."""

from __future__ import annotations

import concurrent.futures
import ctypes
import functools

import numpy as np
import pytest
import torch

from oracle import oracle
from tests.gpu_util import DEV
from tests.test_gpu_solid_maps import CORNER, LENGTH, _scene

pytestmark = pytest.mark.gpu

LEVEL = 9
# name: (seed, cameras, height, width, convention, partial, radius, field of view)
SCENES = {
    "partial cv": (41, 33, 331, 450, "opencv", True, 1.6, 60.0),
    "partial gl": (42, 34, 300, 310, "opengl", True, 1.6, 60.0),
    "70 cv": (43, 70, 200, 260, "opencv", False, 2.5, 40.0),
    "131 gl partial": (44, 131, 190, 180, "opengl", True, 1.6, 60.0),
}


@functools.lru_cache(maxsize=None)
def _case(name):
    seed, cameras, height, width, convention, partial, radius, fovy = SCENES[name]
    masks, T = _scene(seed, cameras, height, width, convention, radius, fovy)
    masks = masks.astype(np.uint8)
    assert cameras << (2 * LEVEL) >= 1 << 23  # the maps are in use
    return masks, T, partial, convention


@functools.lru_cache(maxsize=None)
def _oracle(name):
    masks, T, partial, convention = _case(name)
    return oracle.sparse_field(masks, T, LEVEL, CORNER, LENGTH, partial, convention)


def _stats():
    from torchhull_amd import _lib

    tests, children = (ctypes.c_int64 * 16)(), (ctypes.c_int64 * 16)()
    _lib.check(_lib.lib().thull_visual_hull_stats(_lib.context(0), 16, tests, children))
    return list(tests), list(children)


@pytest.mark.parametrize("name", list(SCENES))
def test_every_launch_shape_equals_the_oracle(name):
    import torchhull_amd as th
    from torchhull_amd import _lib, tuning

    masks, T, partial, convention = _case(name)
    fld = _oracle(name)
    args = (torch.from_numpy(masks).to(DEV), torch.from_numpy(T).to(DEV), LEVEL, CORNER, LENGTH, partial, convention)
    ctx = _lib.context(0)
    saved = tuning.get_carve_tuning(ctx)
    try:
        for lanes in (4, 2, 1):
            print(f"case {name}, {lanes} lanes", flush=True)
            tuning.set_carve_tuning(ctx, tuning._FORCE[lanes])
            cand = th.visual_hull_with_candidate_voxels(*args)[2]
            assert _stats()[0][:len(fld.tests)] == list(fld.tests)
            for i, (a, b) in enumerate(zip(cand, fld.candidates)):
                assert np.array_equal(a.cpu().numpy(), b), f"{lanes} lanes, candidates of level {i}"
            field = th.sparse_visual_hull_field(*args)
            assert np.array_equal(field.values().cpu().numpy().view(np.uint32), fld.values.view(np.uint32))
    finally:
        tuning.set_carve_tuning(ctx, saved)


def _batch(mirror):
    scenes = []
    for name in ("partial cv", "70 cv"):
        masks, T, partial, convention = _case(name)
        T = T * np.array([-1.0 if mirror else 1.0, 1.0, 1.0, 1.0], np.float32)  # the mirrored hull: as large
        scenes.append(dict(masks=torch.from_numpy(masks).to(DEV), transforms=torch.from_numpy(T).to(DEV), level=LEVEL,
                           cube_corner_bfl=CORNER, cube_length=LENGTH, masks_partial=partial,
                           transforms_convention=convention))
    masks, T = _scene(45, 2, 120, 130, "opengl")  # no maps
    scenes.append(dict(masks=torch.from_numpy(masks).to(DEV), transforms=torch.from_numpy(T).to(DEV), level=6,
                       cube_corner_bfl=CORNER, cube_length=LENGTH, masks_partial=False,
                       transforms_convention="opengl"))
    return scenes


def _fresh(f, *args):
    """f in a thread of its own: a new context, which holds no plan of these shapes."""
    with concurrent.futures.ThreadPoolExecutor(1) as pool:
        pool.submit(f, *args).result()


def _replay(lanes):
    import torchhull_amd as th
    from torchhull_amd import _lib, tuning

    ctx = _lib.context(0)
    saved = tuning.get_carve_tuning(ctx)
    try:
        if lanes is not None:
            tuning.set_carve_tuning(ctx, tuning._FORCE[lanes])
        expect = {}
        for mirror in (False, True):
            expect[mirror] = (th.visual_hull_batch(_batch(mirror)), _stats())
        before = th.graph_stats()
        for call, mirror in enumerate((False, False, True, False)):
            print(f"case replay, lanes {lanes}, call {call}", flush=True)
            meshes = th.visual_hull_batch(_batch(mirror), graph=True)
            want, stats = expect[mirror]
            for (v, f), (ev, ef) in zip(meshes, want):
                assert torch.equal(f, ef) and torch.equal(v.view(torch.int32), ev.view(torch.int32))
            assert _stats() == stats
        after = th.graph_stats()
    finally:
        tuning.set_carve_tuning(ctx, saved)
    assert after["captures"] == before["captures"] + 1
    assert after["replays"] - before["replays"] == 3 and after["overflows"] == before["overflows"]


@pytest.mark.parametrize("lanes", [None, 1])
def test_replayed_carving_loop_with_maps_equals_the_host_driven_one(lanes):
    _fresh(_replay, lanes)


def _outgrow():
    import torchhull_amd as th

    big = _batch(False)
    small = [dict(s, masks=torch.zeros_like(s["masks"])) for s in big]
    for s, b in zip(small, big):  # a corner of the masks only: same shapes, far fewer cells
        h, w = b["masks"].shape[1] // 2, b["masks"].shape[2] // 2
        s["masks"][:, h - 6:h + 6, w - 6:w + 6] = b["masks"][:, h - 6:h + 6, w - 6:w + 6]
    print("case overflow", flush=True)
    for _ in range(2):
        th.visual_hull_batch(small, graph=True)
    before = th.graph_stats()
    meshes = th.visual_hull_batch(big, graph=True)
    assert th.graph_stats()["overflows"] == before["overflows"] + 1
    for s, (v, f) in zip(big, meshes):
        ev, ef = th.visual_hull(**s)
        assert torch.equal(f, ef) and torch.equal(v.view(torch.int32), ev.view(torch.int32))


def test_replay_with_maps_that_outgrows_its_plan():
    _fresh(_outgrow)
