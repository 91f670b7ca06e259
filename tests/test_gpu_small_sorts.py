"""The one-launch depth and tile sorts against the oracle (bit-exact order,
offsets, ranges), around the sizes where they change: keys per thread, the
largest primitive and instance counts they take, one and two tile passes, the
largest tile count, equal depths, few visible primitives."""
import dataclasses

import numpy as np
import pytest

from tinygs_amd import scenes

pytestmark = pytest.mark.gpu

# what the one-launch sorts take: primitives (8192, below), instances and tiles
SORT_MAX, TILES_MAX = 16384, 8192


def _scene(n, width, height, scale, seed=31):
    s = scenes.config2(seed=seed, n=n, width=width, height=height)
    means = s.means.copy()
    means[1::7] = means[0]   # equal depths: stable in the index
    return dataclasses.replace(s, means=means, scales=s.scales + np.float32(scale))


def _check(s, orc, image):
    from test_gpu_fgs16 import _check_forward as check16, _render16
    from test_gpu_parity import _check_forward
    return _check_forward(s, orc)[1][1] if image == "float32" else check16(s, orc, _render16(s))[1]


@pytest.mark.parametrize("n", [1, 1023, 1025, 2049, 4096, 4097, 8192, 8193])
def test_depth_counts(hip, orc, n):
    from test_gpu_fgs16 import _check_forward as check16, _render16
    from test_gpu_parity import _check_forward
    s = _scene(n, 300, 213, 0.0)
    _check_forward(s, orc)
    check16(s, orc, _render16(s))


def _sizes(bins):
    return int(bins["n_instances"]), bins["ranges"].size // 2


@pytest.mark.parametrize("width,height,scale", [(64, 64, 0.0), (64, 64, 0.7), (64, 64, 1.2), (64, 64, 2.0),
                                                (1033, 700, -1.0), (1441, 1456, -2.0), (1473, 1473, -2.0)])
def test_instance_and_tile_counts(hip, orc, width, height, scale):
    """16 tiles (one pass), 2860 (two of six bits), and above the largest grid of the one-launch sort."""
    from test_gpu_parity import _check_forward
    s = _scene(1500, width, height, scale)
    _, (pre, bins, fwd) = _check_forward(s, orc)
    instances, tiles = _sizes(bins)
    assert instances <= SORT_MAX and (tiles <= TILES_MAX) == (width < 1400)


@pytest.mark.parametrize("image", ["float32", "float16"])
@pytest.mark.parametrize("width,height", [(2048, 1008), (1440, 1456), (2048, 1024), (2064, 1024)])
def test_tile_limit(hip, orc, width, height, image):
    """8064, 8190 and 8192 tiles (the largest grid of the one-launch sort: passes of six and seven bits), 8256."""
    s = _scene(1500, width, height, -2.0)
    instances, tiles = _sizes(_check(s, orc, image))
    assert instances <= SORT_MAX and (tiles <= TILES_MAX) == (width < 2050) and tiles > 8000


@pytest.mark.parametrize("image", ["float32", "float16"])
@pytest.mark.parametrize("count", [1, 4095, 4096, 4097, 8191, 8192, 8193, 16383, 16384, 16385])
def test_instance_limits(hip, orc, count, image):
    """Exactly that many instances, around the keys per thread of the one-launch tile sort and the most it takes."""
    s = _scene(9000, 300, 213, 0.0)
    nt = (orc.preprocess(s, "f") if image == "float32" else orc.h_preprocess(s))["n_touched"].astype(np.int64)
    keep = (np.cumsum(nt) <= count - min(count, 8)) & (nt > 0)   # the rest of the count in primitives of one tile
    ones = np.flatnonzero((nt == 1) & ~keep)
    keep[ones[:count - nt[keep].sum()]] = True
    means = s.means.copy()
    means[~keep] += np.float32(1e6)
    instances, tiles = _sizes(_check(dataclasses.replace(s, means=means), orc, image))
    assert instances == count and tiles <= TILES_MAX


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


def test_one_rasterizer_through_every_route(hip):
    """Few primitives (waiting: the sort buffers sized by the counts), many, few, no-sync, and few with more instances
    than the one-launch tile sort takes, on one rasterizer: the images of rasterizers of their own."""
    import torch
    from tinygs_amd.core import GPUBatchInput, GPUGaussian3d, Image, RasterizeContext
    from tinygs_amd.rasterizer import create_rasterizer
    few, many, wide = _scene(1200, 131, 77, 0.0), _scene(20000, 131, 77, 0.0), _scene(5000, 300, 213, 1.0)

    def image(r, s, no_sync):
        r.set_gaussians(GPUGaussian3d.from_scene(s))
        ctx = RasterizeContext(fwd_input=GPUBatchInput.from_camera(s.camera))
        ctx.fwd_output.image = Image.empty(s.camera.shape)
        if no_sync:
            r.reserve(100_000, s.camera.grid[0] * s.camera.grid[1])
        r.forward(ctx, no_sync=no_sync)
        torch.cuda.synchronize()
        return ctx.fwd_output.image.data.cpu().numpy(), r.counts()

    r = create_rasterizer("fastgs")
    instances = []
    for s, no_sync in ((few, False), (many, False), (few, False), (many, True), (few, True), (wide, False),
                       (wide, True), (few, False)):
        got, counts = image(r, s, no_sync)
        ref, ref_counts = image(create_rasterizer("fastgs"), s, no_sync)
        assert np.array_equal(got, ref) and counts == ref_counts and r.status() == 0
        instances.append(counts[1])
    assert min(instances) <= SORT_MAX < max(instances) <= 100_000
