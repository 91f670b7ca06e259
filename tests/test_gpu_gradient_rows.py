"""Gradient rows of the preprocess backward at every SH degree and storage type
(each moves another part of the 45-value rows): the assigning backward against
the oracle, and the accumulating one against base + assigned, bit for bit."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("means", "scales", "rotations", "opacities", "sh_coefficient_0", "sh_coefficients_rest")


@pytest.mark.parametrize("sh_dtype", ["float32", "float16"])
@pytest.mark.parametrize("degree", [0, 1, 2, 3])
@pytest.mark.parametrize("n", [257, 1025])
def test_rows_by_degree(hip, orc, n, degree, sh_dtype):
    import torch
    from helpers import assert_grads_close
    from tinygs_amd import scenes
    from tinygs_amd.core import GPUBatchInput, GPUGaussian3d, Image, RasterizeContext
    from tinygs_amd.rasterizer import create_rasterizer
    s = scenes.config2(seed=11, n=n, width=131, height=77)
    s = dataclasses.replace(s, sh_degree=degree, scales=s.scales + np.float32(1.0), sh_dtype=sh_dtype,
                            sh0=s.sh0.astype(np.float16).astype(np.float32),
                            sh_rest=s.sh_rest.astype(np.float16).astype(np.float32))
    gimg = scenes.grad_image(5, s.camera.shape)
    g = GPUGaussian3d.from_scene(s)
    r = create_rasterizer("fastgs")
    r.set_gaussians(g)
    ctx = RasterizeContext(fwd_input=GPUBatchInput.from_camera(s.camera))
    ctx.fwd_output.image = Image.empty(s.camera.shape)
    ctx.grad_output.image = Image(s.camera.shape, "float32", torch.from_numpy(gimg).cuda())
    got = {}
    for assign in (True, False):
        ctx.gaussians_grad = g.gradient_like()
        for t in ctx.gaussians_grad.tensors():
            t.fill_(0.125)
        r.forward(ctx)
        r.backward(ctx, assign=assign)
        torch.cuda.synchronize()
        got[assign] = {f: getattr(ctx.gaussians_grad, f)().cpu().numpy() for f in FIELDS}
    for f in FIELDS:
        assert np.array_equal(np.float32(0.125) + got[True][f], got[False][f]), f
    pre, bins, fwd = orc.render(s, "f")
    ref = orc.preprocess_backward(s, pre, orc.blend_backward(s, pre, bins, fwd, gimg, "f"), "f")
    names = dict(zip(FIELDS, ("means", "scales", "rotations", "opacities", "sh0", "sh_rest")))
    assert_grads_close({names[f]: got[True][f].reshape(-1) for f in FIELDS}, ref)


def test_nan_sigma_weighs_as_the_clamp_does(hip, orc):
    """A Gaussian with a NaN scale reaches the tile of its mean. The backward's clamp max(sigma, 0) takes its sigma
    as 0 (its forward test rejects it), which shows in its colour gradient and those of the Gaussians behind it."""
    import torch
    from helpers import assert_grads_close
    from tinygs_amd import scenes
    from tinygs_amd.core import GPUBatchInput, GPUGaussian3d, Image, RasterizeContext
    from tinygs_amd.rasterizer import create_rasterizer
    s = scenes.config2(seed=11, n=257, width=131, height=77)
    scales = s.scales + np.float32(1.0)
    first = 49   # before the last contributor of its tile (checked below)
    scales[first] = np.nan
    s = dataclasses.replace(s, scales=scales)
    gimg = scenes.grad_image(5, s.camera.shape)
    g = GPUGaussian3d.from_scene(s)
    r = create_rasterizer("fastgs")
    r.set_gaussians(g)
    ctx = RasterizeContext(fwd_input=GPUBatchInput.from_camera(s.camera))
    ctx.fwd_output.image = Image.empty(s.camera.shape)
    ctx.grad_output.image = Image(s.camera.shape, "float32", torch.from_numpy(gimg).cuda())
    ctx.gaussians_grad = g.gradient_like()
    r.forward(ctx)
    r.backward(ctx, assign=True)
    got = {f: getattr(ctx.gaussians_grad, f)().cpu().numpy() for f in FIELDS}
    pre, bins, fwd = orc.render(s, "f")
    assert (bins["inst_prim"] == first).sum() == 1
    ref = orc.preprocess_backward(s, pre, orc.blend_backward(s, pre, bins, fwd, gimg, "f"), "f")
    names = dict(zip(FIELDS, ("means", "scales", "rotations", "opacities", "sh0", "sh_rest")))
    got = {names[f]: got[f].reshape(257, -1).copy() for f in FIELDS}
    ref = {k: ref[k].reshape(257, -1).copy() for k in got}
    assert np.abs(ref["sh0"][first]).max() > 0
    for k in ("means", "scales", "rotations"):   # through the NaN covariance
        got[k][first] = ref[k][first] = 0
    assert_grads_close({k: v.reshape(-1) for k, v in got.items()}, {k: v.reshape(-1) for k, v in ref.items()})
