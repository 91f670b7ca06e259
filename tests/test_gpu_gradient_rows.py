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


def _backwards(s, gimg, image):
    """Gradients (rows, mask, densification info, dL/dw2c) of every backward mode after one forward each."""
    import torch
    from tinygs_amd import _lib
    from tinygs_amd.core import GPUBatchInput, GPUGaussian3d, Image, RasterizeContext
    from tinygs_amd.rasterizer import create_rasterizer
    g = GPUGaussian3d.from_scene(s)
    r = create_rasterizer("fastgs")
    r.set_gaussians(g)
    r.set_params({"enable_pose_opt": True})
    out = {}
    for mode in ("assign", "accumulate", "sparse"):
        ctx = RasterizeContext(fwd_input=GPUBatchInput.from_camera(s.camera))
        ctx.fwd_output.image = Image.empty(s.camera.shape, "cuda", image)
        ctx.grad_output.image = Image(s.camera.shape, image, torch.from_numpy(gimg.astype(image)).cuda())
        if mode == "accumulate":
            ctx.densification_info = torch.zeros((s.n, 4), device="cuda")
        ctx.gaussians_grad = g.gradient_like()
        for t in ctx.gaussians_grad.tensors():
            t.fill_(0.125)
        r.forward(ctx)
        r.backward(ctx, assign=mode == "assign", sparse=mode == "sparse")
        o = {f: getattr(ctx.gaussians_grad, f)().cpu().numpy().reshape(s.n, -1) for f in FIELDS}
        o["w2c"] = np.array(ctx.grad_input.w2c)
        if mode == "accumulate":
            o["info"] = ctx.densification_info.cpu().numpy()
        if mode == "sparse":
            mask = torch.empty(s.n, dtype=torch.uint8, device="cuda")
            _lib.copy_device(r.grad_row_mask(), s.n, mask)
            o["mask"] = mask.cpu().numpy() != 0
        out[mode] = o
    return out


@pytest.mark.parametrize("image", ["float32", "float16"])
@pytest.mark.parametrize("n", [262_145, 300_001, 524_288, 525_001])
def test_rows_of_many_chunks(hip, orc, n, image):
    """Chunks of two and four rounds (the limits are 262,144 and 524,288 primitives; ragged last units): every backward
    mode of a few visible primitives spread over n, against the same primitives alone, bit for bit (a primitive's
    records are summed in one order whatever its chunk). dL/dw2c is regrouped: against the oracle's (float images)
    at the bar of test_gpu_pose.py, and in either type within 1e-4 of the small scene's largest entry (a thread adds
    at most a few terms and the rest is trees of 6, 2 and 8 levels, so about 20 roundings of 2^-24 of the absolute
    sum, 1.2e-6 of it: the bar leaves room for a sum that cancels to 2 %)."""
    from tinygs_amd import scenes
    k = 3000
    s = scenes.config2(seed=11, n=k, width=300, height=213)
    # some hidden, some with more than 16 records
    s = dataclasses.replace(s, scales=s.scales + np.float32(1.5), opacities=s.opacities + np.float32(2.0))
    gimg = scenes.grad_image(5, s.camera.shape)
    if image == "float16":
        gimg = gimg * np.float32(2.0 ** -6)   # sums inside the half range
    idx = np.sort(np.random.default_rng(n).choice(n, k, replace=False))
    idx[0], idx[-1] = 0, n - 1
    w2c = s.camera.w2c
    behind = (s.camera.cam_pos - 5.0 * w2c[2, :3]).astype(np.float32)
    big = {}
    for f in ("means", "scales", "rotations", "opacities", "sh0", "sh_rest"):
        v = getattr(s, f)
        a = np.zeros((n,) + v.shape[1:], np.float32)
        a[...] = behind if f == "means" else v[0]
        a[idx] = v
        big[f] = a
    print(f"[chunks] n={n} {image}", flush=True)
    small = _backwards(s, gimg, image)
    got = _backwards(dataclasses.replace(s, **big), gimg, image)
    rest = np.ones(n, bool)
    rest[idx] = False
    live = small["sparse"]["mask"]
    assert 500 < live.sum() < k
    for mode in ("assign", "accumulate", "sparse"):
        a, b = got[mode], small[mode]
        for f in FIELDS:
            assert np.array_equal(a[f][idx].view(np.uint32), b[f].view(np.uint32)), (mode, f)
            assert np.all(a[f][rest] == (0.0 if mode == "assign" else 0.125)), (mode, f)
        assert np.abs(a["w2c"] - b["w2c"]).max() <= 1e-4 * np.abs(b["w2c"]).max(), mode
    assert np.array_equal(got["sparse"]["mask"][idx], live) and not got["sparse"]["mask"][rest].any()
    # (the forward folds the screen radii, column 3, by groups of 32 neighbours)
    info, alone = got["accumulate"]["info"][:, :3], small["accumulate"]["info"][:, :3]
    assert np.array_equal(info[idx], alone) and not info[rest].any() and (alone[:, 0] > 0).sum() > live.sum()
    if image == "float32":
        from test_gpu_pose import _oracle_pose
        ref, exact = _oracle_pose(orc, s, gimg, "f"), _oracle_pose(orc, s, gimg, "d")
        tol = max(1e-4 * np.abs(exact).max(), 3 * np.abs(ref - exact).max())
        for mode in got:
            assert np.abs(got[mode]["w2c"] - ref).max() <= tol, mode


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
