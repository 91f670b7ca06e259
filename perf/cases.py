"""Timed cases of the FastGS training path, through the package's public entry points.

What a user of this library has it do: train (a TrainStep per view, or the rasterizer / loss / optimizer objects
called one by one as the reference's orchestrator does), differentiate a render, render a view, and call the loss
or the optimizer alone. Scenes are drawn on the GPU with the distributions of tinygs_amd.scenes; the sizes are
those of its configurations, of the tests, or generic ones with odd edges.

Fields of a case:
  kind        "iterate"  TrainStep.step(): forward, fused L1 + SSIM, sparse backward, masked Adam, no host wait
              "contract" the plugin objects in the reference's order: zeroed images and gradients, waiting forward,
                         L1 then SSIM evaluation, accumulating backward, dense Adam
              "gradient" waiting forward, fused L1 + SSIM, assigning backward (with densification info / the pose
                         gradient where the case says so)
              "render"   waiting forward only
              "loss"     fused L1 + SSIM of an image ("assign"), or the two losses accumulated one after the other
              "adam"     one dense SimpleAdam step
  n           Gaussians; width, height: image (absent where the kind has none)
  layout      "ball" (means ~N(0, 1) in a radius-2 ball), "clusters" (32 clusters, 2 % large Gaussians) or
              "cube" (every Gaussian covers many tiles)
  sh_degree, sh ("float32" / "float16" storage), image ("float32" / "float16", the fp16-image rasterizer)
  morton      Gaussians in Morton order, as the training loop leaves them
  info, pose  densification info / the pose gradient asked for
"""
import math

import numpy as np
import torch

from tinygs_amd import create_loss, create_optimizer, create_rasterizer
from tinygs_amd.core import GPUBatchInput, GPUGaussian3d, Image, LossContext, RasterizeContext
from tinygs_amd.image import ImageShape
from tinygs_amd.loss import evaluate_l1_ssim
from tinygs_amd.morton import morton_order
from tinygs_amd.scenes import Camera, Scene, look_at
from tinygs_amd.train import TrainStep

DEVICE = "cuda"
L1_WEIGHT, SSIM_WEIGHT = 0.8, 0.2
# learning-rate factor of the iterated cases: late in a training run, after the exponential schedule's decay
LATE_LR = 0.01
# loss scale of half images, whose gradients (about 1 / pixels) would otherwise be subnormal halves
HALF_SCALE = 4096.0


def _case(name, kind, **kw):
    c = {"name": name, "kind": kind}
    if kind in ("iterate", "contract", "gradient", "render"):
        c.update(n=0, width=0, height=0, layout="ball", sh_degree=3, sh="float32", image="float32", morton=False)
    if kind == "gradient":
        c.update(info=False, pose=False)
    if kind == "loss":
        c.update(width=0, height=0, image="float32", assign=True)
    if kind == "adam":
        c.update(n=0, sh="float32")
    c.update(kw)
    return c


def listed():
    return [
        # a toy scene: every launch is short, so latency and their number count
        _case("toy-1k", "gradient", n=1024, width=64, height=64, sh_degree=0),
        # a small preview in the fp16-image rasterizer, odd size
        _case("preview-half-6k", "render", n=6000, width=246, height=182, image="float16"),
        # an object-sized scene in training
        _case("train-100k", "iterate", n=100_000, width=800, height=800),
        # the headline workload: a large clustered scene with half SH storage
        _case("train-1m", "iterate", n=1_000_000, width=1920, height=1080, layout="clusters", sh="float16"),
        # the same scene in the reference's default training type (half images)
        _case("train-1m-half", "iterate", n=1_000_000, width=1920, height=1080, layout="clusters", sh="float16",
              image="float16"),
        # the training loop's gradients while it densifies: Morton order, densification info
        _case("densify-500k", "gradient", n=500_000, width=1600, height=1060, morton=True, info=True),
        # a caller that keeps to the reference's contract, ragged in every size
        _case("contract-201k", "contract", n=201_377, width=1237, height=823, sh_degree=2),
        # many instances per tile: binning and sorting dominate
        _case("overlap-375k", "gradient", n=375_000, width=3840, height=2160, layout="cube"),
        # evaluation renders of a large scene
        _case("render-1m", "render", n=1_000_003, width=1957, height=1103, layout="clusters"),
        # the losses of a large image in one call, and of half images one by one
        _case("loss-4k", "loss", width=3840, height=2160),
        _case("losses-half", "loss", width=1597, height=1061, image="float16", assign=False),
        # the optimizer on a large scene
        _case("adam-3m", "adam", n=3_000_000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["iterate", "iterate", "contract", "gradient", "gradient", "render", "loss", "adam"])
    c = _case("", kind)
    del c["name"]
    if kind == "adam":
        c.update(n=_log_int(rng, 1000, 3_000_000), sh=rng.choice(["float32", "float16"]))
        return c
    w = _log_int(rng, 64, 3840 if kind == "loss" else 1920)
    c.update(width=w, height=max(48, int(w * rng.uniform(0.5, 1.0))), image=rng.choice(["float32", "float32", "float16"]))
    if kind == "loss":
        c.update(assign=rng.random() < 0.6)
        return c
    layout = rng.choice(["ball", "ball", "clusters", "cube"])
    # at most about one Gaussian per pixel, as scenes in use have
    most = min({"ball": 600_000, "clusters": 1_000_000, "cube": 60_000}[layout], c["width"] * c["height"])
    c.update(layout=layout, n=_log_int(rng, 1000, most),
             sh_degree=rng.choice([0, 1, 2, 3, 3, 3]), sh=rng.choice(["float32", "float16"]),
             morton=rng.random() < 0.4)
    if kind == "gradient":
        c.update(info=rng.random() < 0.5, pose=rng.random() < 0.2)
    return c


# ---------------------------------------------------------------- inputs

def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed) * 7919 + 17)


def _camera(case, seed):
    w, h = case["width"], case["height"]
    v = np.random.default_rng(int(seed)).standard_normal(3)
    v /= np.linalg.norm(v)
    if case["layout"] == "ball":
        return Camera(w, h, 1.375 * w, 1.375 * w, w / 2.0, h / 2.0, look_at(4.0 * v))
    if case["layout"] == "clusters":
        return Camera(w, h, 0.625 * w, 0.625 * w, w / 2.0, h / 2.0, look_at(10.0 * v))
    return Camera(w, h, 2000.0 * w / 3840.0, 2000.0 * w / 3840.0, w / 2.0, h / 2.0, np.eye(4))


def _gaussians(case, seed):
    """Parameter tensors of the case's scene on the device."""
    g = _generator(seed)
    n, layout = case["n"], case["layout"]

    def normal(*shape):
        return torch.randn(*shape, generator=g, device=DEVICE)

    def uniform(*shape):
        return torch.rand(*shape, generator=g, device=DEVICE)

    if layout == "ball":
        means = normal(n, 3)
        means = means * (2.0 / means.norm(dim=1, keepdim=True)).clamp(max=1.0)
        scales, opacities = -4.0 + 0.5 * normal(n, 3), 1.5 * normal(n)
    elif layout == "clusters":
        centres = 6.0 * uniform(32, 3) - 3.0
        which = torch.randint(0, 32, (n,), generator=g, device=DEVICE)
        means = centres[which] + 0.3 * normal(n, 3)
        scales = -4.5 + 0.8 * normal(n, 3)
        scales[uniform(n) < 0.02] = -1.5
        opacities = 0.5 + 1.5 * normal(n)
    else:
        means = uniform(n, 3) - 0.5
        means[:, 2] += 2.0
        scales, opacities = -3.5 + 0.6 * normal(n, 3), -1.0 + normal(n)
    rot = normal(n, 4)
    rot = rot / rot.norm(dim=1, keepdim=True)
    half = torch.float16 if case["sh"] == "float16" else torch.float32
    p = {"means": means, "scales": scales, "rotations": rot, "opacities": opacities,
         "sh0": uniform(n, 3).to(half), "sh_rest": (0.05 * normal(n, 15, 3)).to(half)}
    if case["morton"]:
        order = morton_order(p["means"].contiguous()).long()
        p = {k: v[order] for k, v in p.items()}
    return {k: v.contiguous() for k, v in p.items()}


_FIELDS = {"means": "m_means", "scales": "m_scales", "rotations": "m_rotations", "opacities": "m_opacities",
           "sh0": "m_sh_coefficient_0", "sh_rest": "m_sh_coefficients_rest"}


def _to_gaussian3d(p, sh, degree):
    g = GPUGaussian3d(0, sh, DEVICE)
    for k, f in _FIELDS.items():
        setattr(g, f, p[k])
    g.set_sh_degree(degree)
    return g


def _arrays(g):
    return {k: getattr(g, f) for k, f in _FIELDS.items()}


def _image_type(name):
    return torch.float16 if name == "float16" else torch.float32


def _scale(case):
    return HALF_SCALE if case["image"] == "float16" else 1.0


def _target(shape, seed, dtype):
    g = _generator(seed + 1)
    return torch.rand(shape.padded_size, generator=g, device=DEVICE).to(dtype)


def _pair(case, seed):
    """A target image and a prediction near it, as late in training."""
    shape = ImageShape(case["width"], case["height"], 3)
    target = _target(shape, seed, torch.float32)
    pred = target + 0.1 * torch.randn(shape.padded_size, generator=_generator(seed + 2), device=DEVICE)
    dt = _image_type(case["image"])
    return shape, pred.clamp_(min=0.0).to(dt), target.to(dt)


def _adam_inputs(case, seed):
    """Parameters and the dense gradients of a late step: most rows are zero."""
    p = _gaussians(dict(case, layout="ball", morton=False), seed)
    g = _generator(seed + 3)
    row = (torch.rand(case["n"], generator=g, device=DEVICE) < 0.4).float()
    grads = {}
    for k, v in p.items():
        r = 1e-5 * torch.randn(v.shape, generator=g, device=DEVICE)
        grads[k] = (r * row.view([-1] + [1] * (v.dim() - 1))).contiguous()
    return p, grads


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "loss":
        shape, pred, target = _pair(case, seed)
        dt = case["image"]
        s["ctx"] = LossContext(Image(shape, dt, pred), Image(shape, dt, target), Image.empty(shape, DEVICE, dt),
                               Image.empty(shape, DEVICE, dt))
        s["l1"], s["ssim"] = create_loss("l1"), create_loss("fused_ssim")
        return s
    if kind == "adam":
        p, grads = _adam_inputs(case, seed)
        s["params"] = _to_gaussian3d(p, case["sh"], 3)
        s["opt"] = create_optimizer("simple_adam", s["params"], _to_gaussian3d(grads, "float32", 3))
        return s
    cam = _camera(case, seed)
    p = _gaussians(case, seed)
    target = _target(cam.shape, seed, torch.float32)
    if kind == "iterate":
        host = {k: v.float().cpu().numpy() for k, v in p.items()}
        scene = Scene(host["means"], host["scales"], host["rotations"], host["opacities"], host["sh0"],
                      host["sh_rest"], case["sh_degree"], cam, target.cpu().numpy(), sh_dtype=case["sh"])
        s["train"] = TrainStep(scene, L1_WEIGHT, SSIM_WEIGHT, _scale(case), no_sync=True,
                               image_dtype=case["image"])
        s["train"].optimizer.set_lr(LATE_LR)
        return s
    dt, shape = case["image"], cam.shape
    g = _to_gaussian3d(p, case["sh"], case["sh_degree"])
    r = create_rasterizer("fastgs")
    r.set_gaussians(g)
    ctx = RasterizeContext(fwd_input=GPUBatchInput.from_camera(cam))
    ctx.fwd_output.image = Image.empty(shape, DEVICE, dt)
    s.update(raster=r, ctx=ctx, params=g)
    if kind == "render":
        return s
    ctx.grad_output.image = Image.empty(shape, DEVICE, dt)
    ctx.gaussians_grad = g.gradient_like()
    s["loss"] = LossContext(ctx.fwd_output.image, Image(shape, dt, target.to(_image_type(dt))),
                            Image.empty(shape, DEVICE, dt), ctx.grad_output.image)
    s["l1"], s["ssim"] = create_loss("l1"), create_loss("fused_ssim")
    if kind == "contract":
        s["opt"] = create_optimizer("simple_adam", g, ctx.gaussians_grad)
        s["opt"].set_lr(LATE_LR)
    else:
        r.set_params({"enable_pose_opt": case["pose"]})
        if case["info"]:
            ctx.densification_info = torch.zeros((case["n"], 4), device=DEVICE)
    return s


# ---------------------------------------------------------------- one pass

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "iterate":
        t = state["train"]
        t.step()
        return {"image": t.pred.data, "loss": t.loss_img.data, "grad_image": t.grad_img.data,
                "grads": _arrays(t.grads), "params": _arrays(t.gaussians)}
    if kind == "adam":
        state["opt"].step(1.0)
        return _arrays(state["params"])
    scale = _scale(case)
    if kind == "loss":
        ctx = state["ctx"]
        if case["assign"]:
            evaluate_l1_ssim(state["ssim"], ctx, L1_WEIGHT * scale, SSIM_WEIGHT * scale, assign=True)
        else:
            ctx.loss.data.zero_()
            ctx.grad.data.zero_()
            state["l1"].evaluate(ctx, L1_WEIGHT * scale)
            state["ssim"].evaluate(ctx, SSIM_WEIGHT * scale)
        return {"loss": ctx.loss.data, "grad": ctx.grad.data}
    r, ctx = state["raster"], state["ctx"]
    if kind == "render":
        r.forward(ctx)
        return {"image": ctx.fwd_output.image.data}
    loss = state["loss"]
    if kind == "contract":
        ctx.gaussians_grad.zero_()
        loss.loss.data.zero_()
        loss.grad.data.zero_()
        r.forward(ctx)
        state["l1"].evaluate(loss, L1_WEIGHT * scale)
        state["ssim"].evaluate(loss, SSIM_WEIGHT * scale)
        r.backward(ctx)
        state["opt"].step(1.0 / scale)
        return {"image": loss.pred.data, "loss": loss.loss.data, "grad_image": loss.grad.data,
                "grads": _arrays(ctx.gaussians_grad), "params": _arrays(state["params"])}
    r.forward(ctx)
    evaluate_l1_ssim(state["ssim"], loss, L1_WEIGHT * scale, SSIM_WEIGHT * scale, assign=True)
    r.backward(ctx, assign=True)
    out = {"image": loss.pred.data, "loss": loss.loss.data, "grad_image": loss.grad.data,
           "grads": _arrays(ctx.gaussians_grad)}
    if case["info"]:
        out["info"] = ctx.densification_info
    if case["pose"]:
        out["w2c"] = ctx.grad_input.w2c
    return out


def work(case):
    """Compulsory traffic: parameters, moments and images read and written once, gradients where they are an
    output. Operations: the projection and gradient chain per Gaussian and, per pixel, about 16 blended Gaussians
    until it is opaque; 11 + 11 taps of four (forward) and three (backward) maps for SSIM."""
    kind = case["kind"]
    n = case.get("n", 0)
    px = 3 * case.get("width", 0) * case.get("height", 0)
    e = 2 if case.get("image") == "float16" else 4
    theta = 11 * 4 + 48 * (2 if case.get("sh") == "float16" else 4)
    adam = n * (2 * theta + 4 * 59 * 4)
    ssim_flops = px * 2 * 22 * 7
    if kind == "adam":
        return {"bytes": adam + n * 59 * 4, "flops": n * 59 * 15}
    if kind == "loss":
        return {"bytes": 4 * px * e, "flops": ssim_flops}
    forward = {"bytes": n * theta + px * e, "flops": n * 500 + px // 3 * 16 * 30}
    if kind == "render":
        return forward
    both = {"bytes": forward["bytes"] + 3 * px * e, "flops": 3 * forward["flops"] + ssim_flops}
    if kind == "iterate":
        return {"bytes": both["bytes"] + adam, "flops": both["flops"] + n * 59 * 15}
    if kind == "contract":
        return {"bytes": both["bytes"] + adam + 2 * n * 59 * 4, "flops": both["flops"] + n * 59 * 15}
    return {"bytes": both["bytes"] + n * 59 * 4, "flops": both["flops"]}


def tolerance(case):
    """About four times what other orders of the sums (SSIM taps, the backward's pixel sums) show."""
    kind, half = case["kind"], case.get("image") == "float16"
    if kind == "adam":
        return {"rel": 1e-6, "max": 1e-4}
    if kind in ("loss", "render"):   # half: single roundings of stored values
        return {"rel": 2e-3, "max": 2e-2} if half else {"rel": 1e-5, "max": 1e-3}
    if half:
        return {"rel": 5e-3, "max": 0.9}
    # needle-shaped Gaussians (clusters, cube) multiply the rounding of their 2D sums by their anisotropy
    return {"rel": 1e-4, "max": 2e-2} if case["layout"] == "ball" else {"rel": 3e-3, "max": 0.3}


# ---------------------------------------------------------------- 64-bit results

def exact(case, seed):
    kind = case["kind"]
    if kind == "adam":
        return _exact_adam(*_adam_inputs(case, seed))
    if kind == "loss":
        shape, pred, target = _pair(case, seed)
        loss, grad = _exact_loss(shape, pred.double(), target.double(), _scale(case))
        return {"loss": loss, "grad": grad}
    small = case["n"] <= 4096 and case["width"] * case["height"] <= 256 * 256
    if kind not in ("gradient", "render") or case["image"] != "float32" or not small:
        return None
    cam = _camera(case, seed)
    p = {k: v.double() for k, v in _gaussians(case, seed).items()}
    scene = _ExactScene(p, cam, case["sh_degree"])
    image = scene.forward()
    if kind == "render":
        return {"image": image}
    loss, grad = _exact_loss(cam.shape, image, _target(cam.shape, seed, torch.float32).double())
    out = {"image": image, "loss": loss, "grad_image": grad, "grads": scene.backward(grad)}
    if case["info"]:
        out["info"] = None
    if case["pose"]:
        out["w2c"] = None
    return out


def _exact_adam(p, grads):
    """The first SimpleAdam step from zero moments with the default parameters."""
    lr = {"means": 1.6e-4, "scales": 5e-3, "rotations": 1e-3, "opacities": 5e-2, "sh0": 2.5e-3, "sh_rest": 2.5e-3 * 0.05}
    b1, b2 = 0.9, 0.999
    out = {}
    for k, v in p.items():
        g = grads[k].double().clamp(-1.0, 1.0)
        m, q = (1 - b1) * g, (1 - b2) * g * g
        out[k] = v.double() - lr[k] * (m / (1 - b1)) / ((q / (1 - b2)).sqrt() + 1e-8)
    return out


def _planes(shape, buf):
    """Tiled planar buffer -> (3, padded height, padded width)."""
    t = buf.view(3, shape.tiled_height, shape.tiled_width, 8, 8)
    return t.permute(0, 1, 3, 2, 4).reshape(3, shape.padded_height, shape.padded_width)


def _buffer(shape, planes):
    t = planes.view(3, shape.tiled_height, 8, shape.tiled_width, 8)
    return t.permute(0, 1, 3, 2, 4).reshape(-1)


def _blur(x):
    """11 x 11 Gaussian window, sigma 1.5, zero padding; x: (3, H, W)."""
    i = torch.arange(11, dtype=torch.float64, device=x.device) - 5.0
    w = torch.exp(-i * i / (2 * 1.5 * 1.5))
    w = w / w.sum()
    x = torch.nn.functional.conv2d(x[:, None], w.view(1, 1, 1, 11), padding=(0, 5))
    return torch.nn.functional.conv2d(x, w.view(1, 1, 11, 1), padding=(5, 0))[:, 0]


def _exact_loss(shape, pred, target, scale=1.0):
    """0.8 L1 + 0.2 (1 - SSIM) and its gradient: L1 over the padded image, SSIM statistics from inputs rounded to
    half, its gradient with the unrounded images."""
    w, h = shape.width, shape.height
    p, t = _planes(shape, pred), _planes(shape, target)
    d = p.clamp(0.0, 1.0) - t
    s1, s2 = scale * L1_WEIGHT / (w * h * 3), scale * SSIM_WEIGHT / (w * h)
    loss, grad = d.abs() * s1, torch.where(d >= 0, s1, -s1)
    pi, ti = p[:, :h, :w], t[:, :h, :w]
    x, y = pi.half().double(), ti.half().double()
    mu1, mu2 = _blur(x), _blur(y)
    c1, c2 = 0.01 ** 2, 0.03 ** 2
    a, c = mu1 * mu1 + mu2 * mu2 + c1, 2 * mu1 * mu2 + c1
    b = _blur(x * x + y * y) - mu1 * mu1 - mu2 * mu2 + c2
    e = 2 * (_blur(x * y) - mu1 * mu2) + c2
    loss[:, :h, :w] += (1 - c * e / (a * b)) * s2
    dmu = 2 / (a * b) * (mu2 * (e - c) + mu1 * c * e * (1 / b - 1 / a))
    ds1, ds12 = -c * e / (a * b * b), 2 * c / (a * b)
    grad[:, :h, :w] -= s2 * (_blur(dmu) + 2 * pi * _blur(ds1) + ti * _blur(ds12))
    return _buffer(shape, loss.contiguous()), _buffer(shape, grad.contiguous())


_MIN_ALPHA, _MAX_ALPHA, _T_MIN, _BUCKET = 1.0 / 255.0, 0.999, 1e-4, 32


class _ExactScene:
    """The fp32-image rasterizer of a small scene in 64 bits: every tile's depth-ordered list blended pixel by
    pixel, and the backward's semantics (32-Gaussian buckets restarted from the forward's state, no 1/255 test)."""

    def __init__(self, p, cam, degree):
        self.p = {k: v.detach().clone().requires_grad_(True) for k, v in p.items()}
        self.cam, self.degree = cam, degree
        dev = p["means"].device
        self.w2c = torch.tensor(np.asarray(cam.w2c, np.float32), dtype=torch.float64, device=dev)
        self.cam_pos = torch.tensor(np.asarray(cam.cam_pos, np.float64), device=dev)
        self._project()

    def _project(self):
        cam, p, w = self.cam, self.p, self.w2c
        f32 = lambda v: float(np.float32(v))   # noqa: E731  the camera arrives in float
        fx, fy, cx, cy = f32(cam.fx), f32(cam.fy), f32(cam.cx), f32(cam.cy)
        t = p["means"] @ w[:3, :3].T + w[:3, 3]
        z = t[:, 2]
        q = p["rotations"] / p["rotations"].norm(dim=1, keepdim=True)
        r, x, y, v = q.unbind(1)
        rot = torch.stack([1 - 2 * (y * y + v * v), 2 * (x * y - r * v), 2 * (x * v + r * y),
                           2 * (x * y + r * v), 1 - 2 * (x * x + v * v), 2 * (y * v - r * x),
                           2 * (x * v - r * y), 2 * (y * v + r * x), 1 - 2 * (x * x + y * y)], 1).view(-1, 3, 3)
        m = rot * p["scales"].exp()[:, None, :]
        cov = m @ m.transpose(1, 2)
        ux, uy = t[:, 0] / z, t[:, 1] / z

        def clamped(u, size, c, f):   # the Jacobian's frustum clamp: no gradient past it
            lo, hi = (-0.15 * size - c) / f, (1.15 * size - c) / f
            return u.clamp(lo, hi), (u > lo) & (u < hi)

        tx, okx = clamped(ux, cam.width, cx, fx)
        ty, oky = clamped(uy, cam.height, cy, fy)
        j11, j22 = fx / z, fy / z
        j13, j23 = -fx / z * tx, -fy / z * ty
        j13, j23 = torch.where(okx, j13, j13.detach()), torch.where(oky, j23, j23.detach())
        zero = torch.zeros_like(z)
        jac = torch.stack([torch.stack([j11, zero, j13], 1), torch.stack([zero, j22, j23], 1)], 1) @ w[:3, :3]
        c2 = jac @ cov @ jac.transpose(1, 2)
        a, b, c = c2[:, 0, 0] + 0.3, c2[:, 0, 1], c2[:, 1, 1] + 0.3
        det = a * c - b * b
        self.mean2d = torch.stack([ux * fx + cx, uy * fy + cy], 1)
        self.conic = torch.stack([c / det, -b / det, a / det], 1)
        self.opacity = torch.sigmoid(p["opacities"])
        self.color = self._colors()
        with torch.no_grad():
            thr = torch.log(self.opacity * 255.0)
            ok = (z >= cam.near) & (z <= cam.far) & (self.opacity >= _MIN_ALPHA) & (det >= 1e-8)
            fac = (2.0 * thr.clamp(min=0.0)).sqrt()
            ext = torch.stack([(fac * a.sqrt() - 0.5).clamp(min=0.0), (fac * c.sqrt() - 0.5).clamp(min=0.0)], 1)
            self.lo = ((self.mean2d - ext) / 16.0).floor()
            self.hi = ((self.mean2d + ext) / 16.0).ceil()
            self.thr, self.ok, self.z = thr, ok, z

    def _colors(self):
        p, deg = self.p, self.degree
        d = p["means"] - self.cam_pos
        x, y, z = (d / d.norm(dim=1, keepdim=True)).unbind(1)
        k = []
        if deg > 0:
            k += [-0.48860251190291987 * y, 0.48860251190291987 * z, -0.48860251190291987 * x]
        if deg > 1:
            k += [1.0925484305920792 * x * y, -1.0925484305920792 * y * z,
                  0.94617469575755997 * z * z - 0.31539156525251999, -1.0925484305920792 * x * z,
                  0.54627421529603959 * (x * x - y * y)]
        if deg > 2:
            k += [0.59004358992664352 * y * (y * y - 3 * x * x), 2.8906114426405538 * x * y * z,
                  0.45704579946446572 * y * (1 - 5 * z * z), 0.3731763325901154 * z * (5 * z * z - 3),
                  0.45704579946446572 * x * (1 - 5 * z * z), 1.4453057213202769 * z * (x * x - y * y),
                  0.59004358992664352 * x * (3 * y * y - x * x)]
        c = 0.5 + 0.28209479177387814 * p["sh0"]
        for i, b in enumerate(k):
            c = c + b[:, None] * p["sh_rest"][:, i]
        return c

    def _lists(self):
        """(tiles, longest list) primitive indices in depth order, -1 past a tile's end."""
        cam = self.cam
        gw, gh = cam.grid
        dev = self.z.device
        tiles = torch.arange(gw * gh, device=dev)
        tx, ty = (tiles % gw)[:, None].double(), (tiles // gw)[:, None].double()
        hit = self.ok & (self.lo[:, 0] <= tx) & (tx < self.hi[:, 0]) & (self.lo[:, 1] <= ty) & (ty < self.hi[:, 1])
        mx, my = self.mean2d[:, 0] - 0.5, self.mean2d[:, 1] - 0.5
        a, b, c = self.conic.unbind(1)
        x0, y0 = tx * 16, ty * 16
        x1, y1 = x0 + 15, y0 + 15
        left, above = (x0 > mx), (y0 > my)
        out_x, out_y = left | (mx > x1), above | (my > y1)
        qx, qy = torch.where(left, x0, x1), torch.where(above, y0, y1)
        fx, fy = mx - qx, my - qy
        dx, dy = torch.where(x0 - mx >= 0, 15.0, -15.0), torch.where(y0 - my >= 0, 15.0, -15.0)
        ux = out_y * ((dx * a * fx + dx * b * fy) / (dx * a * dx)).clamp(0, 1)
        uy = out_x * ((dy * b * fx + dy * c * fy) / (dy * c * dy)).clamp(0, 1)
        gx, gy = mx - (qx + ux * dx), my - (qy + uy * dy)
        power = 0.5 * (a * gx * gx + c * gy * gy) + b * gx * gy
        hit &= ~(out_x | out_y) | (power <= self.thr)
        order = torch.argsort(self.z.float(), stable=True)
        hit = hit[:, order]
        k = int(hit.sum(1).max())
        pos = hit.cumsum(1) - 1
        idx = torch.full((gw * gh, max(k, 1)), -1, dtype=torch.long, device=dev)
        t, j = hit.nonzero(as_tuple=True)
        idx[t, pos[t, j]] = order[j]
        return idx

    @torch.no_grad()
    def forward(self):
        cam, shape = self.cam, self.cam.shape
        gw, gh = cam.grid
        dev = self.z.device
        self.idx = self._lists()
        tiles = torch.arange(gw * gh, device=dev)
        i = torch.arange(256, device=dev)
        self.px = (tiles % gw)[:, None] * 16 + i % 16
        self.py = (tiles // gw)[:, None] * 16 + i // 16
        self.inside = (self.px < cam.width) & (self.py < cam.height)
        T = self.inside.double()
        C = torch.zeros(*T.shape, 3, dtype=torch.float64, device=dev)
        self.last = torch.zeros(T.shape, dtype=torch.long, device=dev)
        self.states = []
        for k in range(self.idx.shape[1]):
            if k % _BUCKET == 0:
                self.states.append((C.clone(), T.clone()))
            sigma, X, Y, op, col, _ = self._pair(k)
            alpha = (op * torch.exp(-sigma)).clamp(max=_MAX_ALPHA)
            ok = (sigma >= 0) & (alpha >= _MIN_ALPHA) & (self.idx[:, k] >= 0)[:, None]
            nT = T * (1 - alpha)
            keep = ok & (nT >= _T_MIN)
            C = C + torch.where(keep, T * alpha, 0.0)[..., None] * col[:, None]
            T = torch.where(ok, torch.where(keep, nT, 0.0), T)
            self.last = torch.where(keep, k + 1, self.last)
        self.out = C
        planes = torch.zeros(3, gh * 16, gw * 16, dtype=torch.float64, device=dev)
        planes[:, self.py, self.px] = torch.where(self.inside[..., None], C, 0.0).permute(2, 0, 1)
        return _buffer(shape, planes[:, :shape.padded_height, :shape.padded_width].contiguous())

    def _pair(self, k):
        p = self.idx[:, k].clamp(min=0)
        m, con = self.mean2d.detach()[p], self.conic.detach()[p]
        X, Y = m[:, :1] - (self.px + 0.5), m[:, 1:] - (self.py + 0.5)
        sigma = 0.5 * (con[:, :1] * X * X + con[:, 2:] * Y * Y) + con[:, 1:2] * X * Y
        return sigma, X, Y, self.opacity.detach()[p][:, None], self.color.detach()[p].clamp(min=0.0), con

    def backward(self, grad_buffer):
        n, dev = self.z.shape[0], self.z.device
        shape = self.cam.shape
        gw, gh = self.cam.grid
        planes = torch.zeros(3, gh * 16, gw * 16, dtype=torch.float64, device=dev)
        planes[:, :shape.padded_height, :shape.padded_width] = _planes(shape, grad_buffer)
        g = planes[:, self.py, self.px].permute(1, 2, 0)
        g = torch.where(self.inside[..., None], g, 0.0)
        sums = torch.zeros(n, 9, dtype=torch.float64, device=dev)
        for k in range(self.idx.shape[1]):
            if k % _BUCKET == 0:
                C, T = self.states[k // _BUCKET]
                rest = ((self.out - C) * g).sum(-1)
            sigma, X, Y, op, col, con = self._pair(k)
            on = (k < self.last) & (self.idx[:, k] >= 0)[:, None]
            alpha = (op * torch.exp(-sigma.clamp(min=0.0))).clamp(max=_MAX_ALPHA)
            wgt = torch.where(on, T * alpha, 0.0)
            cg = (col[:, None] * g).sum(-1)
            rest = rest - wgt * cg
            pp = torch.where(on, alpha * (T * cg - rest / (1 - alpha)), 0.0)
            T = torch.where(on, T * (1 - alpha), T)
            a, b, c = con[:, :1], con[:, 1:2], con[:, 2:]
            each = torch.stack([(-pp * (a * X + b * Y)).sum(1), (-pp * (b * X + c * Y)).sum(1),
                                (-0.5 * pp * X * X).sum(1), (-pp * X * Y).sum(1), (-0.5 * pp * Y * Y).sum(1),
                                (wgt * g[..., 0]).sum(1), (wgt * g[..., 1]).sum(1), (wgt * g[..., 2]).sum(1),
                                pp.sum(1)], 1)
            here = self.idx[:, k] >= 0
            sums.index_add_(0, self.idx[here, k], each[here])
        color_grad = torch.where(self.color >= 0, sums[:, 5:8], 0.0)
        torch.autograd.backward([self.mean2d, self.conic, self.color], [sums[:, :2], sums[:, 2:5], color_grad])
        out = {k: (v.grad if v.grad is not None else torch.zeros_like(v)) for k, v in self.p.items()}
        out["opacities"] = sums[:, 8] * (1 - self.opacity.detach())
        return out
