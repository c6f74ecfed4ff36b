"""Solid maps of masks whose integral images round: values well above 1 beside the solid regions, with totals that
leave windows a small reach (torchhull_amd/csrc/solid_reach.h), against the oracle."""

from __future__ import annotations

import numpy as np
import pytest

from tests.test_gpu_solid_maps import _check, _scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [1.3, 5.7, 21.9])
@pytest.mark.parametrize("partial", [False, True])
def test_fractions_above_one_beside_solid_regions(scale, partial):
    masks, T = _scene(31, 36, 320, 322, "opengl")
    rng = np.random.default_rng(32)
    # inside the silhouettes: bands of large fractions, so that the rest of each row and column sums past them
    bright = (scale * (0.5 + rng.random(masks.shape))).astype(np.float32)
    band = np.zeros(masks.shape, dtype=bool)
    band[:, :, 120:128] = True
    band[:, 110:114] = True
    masks = np.where(band & (masks == 1.0), bright, masks)
    print(f"case fractions scale={scale} partial={partial}", flush=True)
    assert _check(masks, T, 9, partial, "opengl") > 1000
