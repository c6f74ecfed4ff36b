"""Blur kernel sizes around the compiled tap counts and the groups of 8 taps of the other sizes, on images whose
edges cut the 64-pixel blocks: band blur bit for bit against the oracle, dense blur against float64."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle
from tests.gpu_util import DEV

pytestmark = pytest.mark.gpu


def _image(seed: int, B: int, H: int, W: int) -> np.ndarray:
    rng = np.random.default_rng(seed)
    im = np.zeros((B, H, W, 1), np.uint8)
    y, x = np.mgrid[:H, :W]
    for b in range(B):
        for _ in range(3):
            cy, cx, r = rng.uniform(0, H), rng.uniform(0, W), rng.uniform(3, 0.4 * max(H, W))
            im[b, :, :, 0] |= ((y - cy) ** 2 + (x - cx) ** 2 < r * r).astype(np.uint8)
    return im


@pytest.mark.parametrize("k", [11, 13, 17, 19, 23, 25])
@pytest.mark.parametrize("in_dtype", [np.float32, np.uint8, np.float64])
@pytest.mark.parametrize("out_dtype", [np.float16, np.float32, np.float64])
def test_band_blur_tap_groups_match_oracle(k, in_dtype, out_dtype):
    import torchhull_amd as th

    im = _image(k, 2, 77, 131).astype(in_dtype)
    td = {np.float16: torch.float16, np.float32: torch.float32, np.float64: torch.float64}[out_dtype]
    print(f"case k={k} {in_dtype.__name__} -> {out_dtype.__name__}", flush=True)
    got = th.gaussian_blur(torch.from_numpy(im).to(DEV), k, 2.1, sparse=True, dtype=td).cpu().numpy()
    ref = oracle.gaussian_blur_sparse(im, k, 2.1, out_dtype)
    assert np.array_equal(got.view(np.uint8), ref.view(np.uint8))


@pytest.mark.parametrize("k", [11, 13, 17, 23])
@pytest.mark.parametrize("shape", [(1, 64, 64), (2, 65, 130), (1, 40, 200)])
def test_dense_blur_tap_groups_match_float64(k, shape):
    import torchhull_amd as th

    sigma, h = 2.1, k // 2
    x = torch.from_numpy(np.random.default_rng(k).uniform(0, 1, size=(*shape, 1)).astype(np.float32))
    got = th.gaussian_blur(x.to(DEV), k, sigma, sparse=False, dtype=torch.float32).cpu()[..., 0].double()
    t = torch.arange(-h, h + 1, dtype=torch.float64)
    w = torch.exp(-(t[:, None] ** 2 + t[None, :] ** 2) / (2.0 * sigma ** 2))
    pad = torch.nn.functional.pad(x[..., 0].double()[:, None], (h, h, h, h), mode="reflect")
    ref = torch.nn.functional.conv2d(pad, (w / w.sum())[None, None])[:, 0]
    # k^2 fused multiply-adds of values up to 1, and weights normalised by a sequential float32 sum of k^2 terms:
    # each contributes at most k^2 + 2 roundings of 2^-24
    assert (got - ref).abs().max() <= 2 * (k * k + 2) * 2.0 ** -24
