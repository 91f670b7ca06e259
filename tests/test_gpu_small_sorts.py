"""The one-launch depth and tile sorts against the oracle (bit-exact order,
offsets, ranges), around the sizes where they change: keys per thread, the
largest primitive and instance counts they take, one and two tile passes, the
largest tile count, equal depths, few or no visible primitives."""
import dataclasses

import numpy as np
import pytest

from tinygs_amd import scenes

pytestmark = pytest.mark.gpu


def _scene(n, width, height, scale, seed=31):
    s = scenes.config2(seed=seed, n=n, width=width, height=height)
    means = s.means.copy()
    means[1::7] = means[0]   # equal depths: stable in the index
    return dataclasses.replace(s, means=means, scales=s.scales + np.float32(scale))


@pytest.mark.parametrize("n", [1, 1023, 1025, 2049, 4096, 4097, 8192, 8193])
def test_depth_counts(hip, orc, n):
    from test_gpu_fgs16 import _check_forward as check16, _render16
    from test_gpu_parity import _check_forward
    s = _scene(n, 300, 213, 0.0)
    _check_forward(s, orc)
    check16(s, orc, _render16(s))


@pytest.mark.parametrize("width,height,scale", [(64, 64, 0.0), (64, 64, 0.7), (64, 64, 1.2), (64, 64, 2.0),
                                                (1033, 700, -1.0), (1441, 1456, -2.0), (1473, 1473, -2.0)])
def test_instance_and_tile_counts(hip, orc, width, height, scale):
    from test_gpu_parity import _check_forward
    s = _scene(1500, width, height, scale)
    _, (pre, bins, fwd) = _check_forward(s, orc)
    print("instances", bins["n_instances"], "tiles", bins["ranges"].size // 2, flush=True)


def test_few_visible(hip, orc):
    from test_gpu_parity import _check_forward
    s = _scene(3000, 131, 77, 0.0)
    means = s.means.copy()
    means[np.arange(3000) != 1777] += np.float32(1e6)
    run, (pre, bins, fwd) = _check_forward(dataclasses.replace(s, means=means), orc)
    assert bins["n_visible"] == 1


def test_no_sync_forward_matches_waiting(hip):
    """The instance count on the device, the capacity one that the one-launch tile sort takes or not."""
    import torch
    from tinygs_amd.core import GPUBatchInput, GPUGaussian3d, Image, RasterizeContext
    from tinygs_amd.rasterizer import create_rasterizer
    s = _scene(1200, 131, 77, 0.0)
    images = []
    for cap in (None, 16384, 16385):
        r = create_rasterizer("fastgs")
        r.set_gaussians(GPUGaussian3d.from_scene(s))
        ctx = RasterizeContext(fwd_input=GPUBatchInput.from_camera(s.camera))
        ctx.fwd_output.image = Image.empty(s.camera.shape)
        if cap:
            r.reserve(cap, s.camera.grid[0] * s.camera.grid[1])
        for _ in range(2):
            r.forward(ctx, no_sync=cap is not None)
        torch.cuda.synchronize()
        assert r.status() == 0
        images.append(ctx.fwd_output.image.data.cpu().numpy())
    assert np.array_equal(images[0], images[1]) and np.array_equal(images[0], images[2])
