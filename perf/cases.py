"""What a program does with this rasterizer, as cases to time: rendering a cloud
(to host memory, or into GPU memory without allocating), computing gradients,
and training on one view or several, over the sizes, SH degrees and storages,
sum kinds, tile shapes and scene statistics that the benchmark workloads
(vsplat.fixtures.config) and the tests use.

A case is a dict: `call` names the entry points (see run), the rest the scene
and the trainer's options. prepare() makes what such a program holds before the
call, run() is one pass, exact() the same outputs in 64-bit floats.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.getcwd(), "vibe-splat_amd"))  # the package's folder, in the repository's root
import vsplat  # noqa: E402
from vsplat.fixtures import Camera, Cloud  # noqa: E402

TILES = {"16x16": vsplat.TILES_16X16, "8x8": vsplat.TILES_8X8, "32x8": vsplat.TILES_32X8, "32x32": vsplat.TILES_32X32}
# A ring of eight views of uneven size, as one training batch sees a scene.
RING = ((640, 480), (960, 540), (1280, 720), (1280, 720), (1280, 720), (1600, 900), (1920, 1080), (1920, 1080))
# Learning rates late in training: the position's is where the usual schedule
# ends; the others are lowered alike, so that many steps leave the scene's
# statistics as they are.
RATES = vsplat.LearningRates(position=1.6e-6, scale=1e-4, rotation=2e-5, opacity=1e-3, sh=5e-4, sh_rest_scale=0.05)

DEFAULTS = {"degree": 3, "scene": "uniform", "bf16": False, "fixed": False, "tiles": "16x16", "lambda": 0.2, "mip": False,
            "recompute": False, "penalties": 0.0, "views": 1}


def listed():
    return [
        # A preview of a small cloud: launches and latency.
        {"name": "preview", "call": "render", "n": 10_000, "degree": 0, "width": 256, "height": 256},
        # The smallest training workload, L1 only, its gradients read by an optimiser on the host.
        {"name": "gradients", "call": "gradients", "n": 10_000, "degree": 0, "width": 256, "height": 256, "lambda": 0.0},
        # Gradients summed over three odd-sized views, read on the host.
        {"name": "accumulate", "call": "accumulate", "n": 40_000, "degree": 2, "width": 333, "height": 251, "views": 3, "fixed": True},
        # Serving: a cloud of the allocation-free render's size into a GPU buffer.
        {"name": "serve", "call": "noalloc", "n": 100_000, "width": 1280, "height": 720},
        # A held-out view rendered to host memory for an image metric; odd size, Mip-Splatting's 2D filter.
        {"name": "evaluate", "call": "render", "n": 300_000, "width": 979, "height": 733, "mip": True},
        # The start of a training run: few Gaussians, a small image, MCMC's penalties.
        {"name": "train early", "call": "step", "n": 30_000, "width": 640, "height": 480, "penalties": 0.01},
        # The headline workload as a training step: target from the host, loss back, each call waited for.
        {"name": "train", "call": "step", "n": 1_000_000, "width": 1280, "height": 720, "fixed": True, "tiles": "32x32"},
        # Steps queued back to back against targets on the GPU; odd size, bf16 SH, float sums.
        {"name": "train queued", "call": "queue", "n": 400_000, "width": 1001, "height": 667, "bf16": True},
        # A large clustered scene at 1920x1080.
        {"name": "train large", "call": "step", "n": 3_000_000, "width": 1920, "height": 1080, "scene": "blobs", "bf16": True,
         "fixed": True, "tiles": "32x32"},
        # Heavy-tailed sizes: long lists; the backward recomputes the transmittance.
        {"name": "train heavy", "call": "step", "n": 1_000_000, "degree": 2, "width": 1920, "height": 1080, "scene": "heavy",
         "fixed": True, "tiles": "32x32", "recompute": True},
        # Eight views of uneven size a step, captured once as a graph and replayed.
        {"name": "train batch", "call": "captured", "n": 1_000_000, "width": 0, "height": 0, "views": 8, "bf16": True, "fixed": True,
         "tiles": "32x32"},
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    call = rng.choice(("render", "gradients", "accumulate", "noalloc", "step", "step", "queue", "captured"))
    scene = rng.choice(("uniform", "uniform", "blobs", "heavy"))
    case = {"call": call, "scene": scene, "degree": rng.randint(0, 3), "width": _log_uniform(rng, 96, 1920),
            "height": _log_uniform(rng, 96, 1080), "bf16": rng.random() < 0.4, "fixed": rng.random() < 0.5,
            "tiles": rng.choice(tuple(TILES)), "lambda": rng.choice((0.0, 0.2, 0.2)), "mip": rng.random() < 0.25,
            "recompute": rng.random() < 0.25, "penalties": rng.choice((0.0, 0.0, 0.01))}
    most = {"gradients": 60_000, "accumulate": 60_000, "noalloc": 120_000, "captured": 400_000}.get(call, 1_000_000)
    if scene == "heavy":
        most = min(most, 300_000)
    if call == "noalloc":  # within its limits on tile entries
        case.update(scene="uniform" if scene == "heavy" else scene, tiles="16x16")
    case["n"] = _log_uniform(rng, 2_000, most)
    case["views"] = rng.randint(2, 5) if call in ("accumulate", "captured") else 1
    return case


# ---------------------------------------------------------------- inputs

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _cloud_arrays(case, seed):
    """positions, log-scales, rotations, opacity logits and SH as float32 tensors: the
    benchmark clouds' distributions. The SH values are ones its storage holds, as those
    of a cloud in training are."""
    c = {**DEFAULTS, **case}
    device = _device()
    g = torch.Generator(device=device).manual_seed(seed * 1_000_003 + 17)
    n, k = c["n"], (c["degree"] + 1) ** 2

    def uniform(*shape):
        return torch.rand(shape, generator=g, device=device)

    def normal(*shape):
        return torch.randn(shape, generator=g, device=device)

    if c["scene"] == "blobs":
        centres = uniform(64, 3) * 2 - 1
        positions = centres[torch.randint(64, (n,), generator=g, device=device)] + 0.2 * normal(n, 3)
    else:
        positions = uniform(n, 3) * 2 - 1
    mean, spread, logit, logit_spread = (-3.5, 1.2, 1.0, 1.5) if c["scene"] == "heavy" else (-4.0, 0.5, 0.0, 1.0)
    scales = mean + spread * normal(n, 3)
    rotations = torch.nn.functional.normalize(normal(n, 4), dim=1)
    opacities = logit + logit_spread * normal(n)
    if k == 1:
        sh = (uniform(n, 1, 3) - 0.5) / 0.28209479177387814
    else:
        sh = 0.3 * normal(n, k, 3)
    if c["bf16"]:
        sh = sh.bfloat16().float()
    else:
        sh[:, 1:] = sh[:, 1:].half().float()
    return positions, scales, rotations, opacities, sh


def _cameras(case):
    """Cameras on a ring of radius 3 about the origin, the first on the z axis."""
    c = {**DEFAULTS, **case}
    sizes = RING[:c["views"]] if c["width"] == 0 else [(c["width"] + 8 * k, c["height"] + 5 * k) for k in range(c["views"])]
    cameras = []
    for k, (w, h) in enumerate(sizes):
        th = 2 * math.pi * k / c["views"]
        eye = np.array([3 * math.sin(th), 0.0, -3 * math.cos(th)])
        forward = -eye / np.linalg.norm(eye)
        right = np.cross([0.0, 1.0, 0.0], forward)
        right /= np.linalg.norm(right)
        view = np.eye(4)
        view[:3, :3] = np.stack([right, np.cross(forward, right), forward])
        view[:3, 3] = -view[:3, :3] @ eye
        f = 0.5 * h / math.tan(math.radians(60.0) / 2)
        f = float(np.float32(f))
        cameras.append(Camera(view=view.astype(np.float32), position=eye.astype(np.float32), fx=f, fy=f, cx=0.5 * w, cy=0.5 * h,
                              width=w, height=h))
    return cameras


def _target(camera, seed):
    """A smooth RGBA8 image with a little noise."""
    rng = np.random.default_rng(seed)
    w, h = camera.width, camera.height
    x, y = np.arange(w, dtype=np.float32)[None, :], np.arange(h, dtype=np.float32)[:, None]
    noise = rng.integers(0, 16, (h, w, 2), dtype=np.uint8)
    out = np.empty((h, w, 4), np.uint8)
    out[..., 0] = (127.0 + 100.0 * np.sin(0.2 * x)).astype(np.uint8) + noise[..., 0]
    out[..., 1] = (127.0 + 100.0 * np.cos(0.15 * y)).astype(np.uint8) + noise[..., 1]
    out[..., 2] = (60 + (x + y) % 120).astype(np.uint8)
    out[..., 3] = 255
    return out


class _DeviceView:
    """Device memory for torch to look at; holds the object that owns it."""

    def __init__(self, owner, pointer, shape, typestr, strides=None):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (pointer, False), "strides": strides, "version": 2}

    def tensor(self):
        return torch.as_tensor(self, device="cuda")


def _parameter_views(trainer, case):
    """The trainer's parameters as tensors on its own buffers (vsplat_parameters' layout)."""
    n, k = trainer.count, (trainer.sh_degree + 1) ** 2
    views = {}
    for group, (name, shape) in enumerate((("positions", (n, 3)), ("scales", (n, 3)), ("rotations", (n, 4)), ("opacities", (n,)))):
        views[name] = _DeviceView(trainer, trainer.parameters(group)[0], shape, "<f4").tensor()
    pointer, size = trainer.parameters(4)
    words = size // (4 * n)
    if case["bf16"]:
        values = _DeviceView(trainer, pointer, (n, 2 * words), "<i2").tensor().view(torch.bfloat16)
        views["sh"] = values[:, :3 * k]
    else:
        views["sh_dc"] = _DeviceView(trainer, pointer, (n, 3), "<f4", (4 * words, 4)).tensor()
        if k > 1:
            views["sh_rest"] = _DeviceView(trainer, pointer + 12, (n, 3 * k - 3), "<f2", (4 * words, 2)).tensor()
    return views


def prepare(case, seed):
    c = {**DEFAULTS, **case}
    arrays = [a.cpu().numpy() for a in _cloud_arrays(c, seed)]
    cloud = Cloud(*arrays, c["degree"])
    options = vsplat.TrainerOptions(lambda_ssim=c["lambda"], force_fixed_point=c["fixed"], mip_filter_2d=c["mip"],
                                    sh_storage=vsplat.SH_BF16 if c["bf16"] else vsplat.SH_HALF, tile_shape=TILES[c["tiles"]],
                                    recompute_transmittance=c["recompute"], opacity_reg=c["penalties"], scale_reg=c["penalties"])
    trainer = vsplat.Trainer(cloud, options)
    cameras = _cameras(c)
    state = {"call": c["call"], "trainer": trainer, "cameras": cameras}
    if c["call"] == "render":
        trainer.render(cameras[0])  # the buffers for this size
        return state
    if c["call"] == "noalloc":
        w, h = cameras[0].width, cameras[0].height
        out = state["out"] = vsplat.DeviceBuffer.empty(w * h * 16)
        state["image"] = _DeviceView(out, out.ptr, (h, w, 4), "<f4").tensor()
        return state
    state["targets"] = targets = [_target(camera, seed * 64 + k) for k, camera in enumerate(cameras)]
    if c["call"] in ("gradients", "accumulate"):
        return state
    state["parameters"] = _parameter_views(trainer, c)
    if c["call"] == "step":
        return state
    # Queued steps do not grow the tile lists: one waited-for pass sizes them.
    state["device"] = [vsplat.DeviceBuffer(t) for t in targets]
    if c["call"] == "queue":
        trainer.set_stage_timing(False)
        trainer.compute_gradients(cameras[0], targets[0])
    else:
        trainer.step_views(cameras, targets)
        trainer.capture_views(cameras, [d.ptr for d in state["device"]], vsplat.MODE_STEP, RATES)
    return state


def _stats(s):
    return {"loss": s.loss, "l1": s.l1, "ssim": s.ssim, "visible": s.visible_splats}


def _gradients(trainer):
    g = trainer.gradients()
    return {"positions": g.positions, "scales": g.scales, "rotations": g.rotations, "opacities": g.opacities, "sh": g.sh}


def run(state):
    call, trainer, cameras = state["call"], state["trainer"], state["cameras"]
    if call == "render":
        return trainer.render(cameras[0])
    if call == "noalloc":
        trainer.render_noalloc(cameras[0], state["out"])
        return state["image"]
    if call == "gradients":
        stats = trainer.compute_gradients(cameras[0], state["targets"][0])
        return {"stats": _stats(stats), "gradients": _gradients(trainer)}
    if call == "accumulate":
        stats = trainer.step_views(cameras, state["targets"])
        return {"stats": [_stats(s) for s in stats], "gradients": _gradients(trainer)}
    if call == "step":
        target = state["targets"][0]
        stats = trainer.step(cameras[0], target, RATES, next_target=target)
        return {"stats": _stats(stats), "parameters": state["parameters"]}
    if call == "queue":
        trainer.enqueue(cameras[0], state["device"][0].ptr, vsplat.MODE_STEP, RATES)
    else:
        trainer.launch_captured(1)
    return {"parameters": state["parameters"]}


def work(case):
    """Bytes: the parameters read, the image or the target, and what is written:
    gradients, or the parameters and two 16-bit Adam moments each, read and written.
    Operations: per Gaussian and view the projection, the colour and (backward) their
    derivatives; per pixel the 11-tap windows of the loss; per pixel and splat in front of
    its stop (at most about 55 with these opacities) the blending and its derivative."""
    c = {**DEFAULTS, **case}
    n, k = c["n"], (c["degree"] + 1) ** 2
    sh = 6 * k if c["bf16"] else 12 + 6 * (k - 1)
    stored, floats = 44 + sh, 11 + 3 * k
    pixels = [cam.width * cam.height for cam in _cameras(c)]
    backward = c["call"] not in ("render", "noalloc")
    moved = n * stored
    if not backward:
        moved += 16 * pixels[0]
    else:
        moved += 4 * sum(pixels)
        moved += 4 * n * floats if c["call"] in ("gradients", "accumulate") else n * (stored + 8 * floats)
    flops = 0.0
    for cam, p in zip(_cameras(c), pixels):
        sigma = (0.06 if c["scene"] == "heavy" else 0.02) * cam.fy / 3
        pairs = p * min(55.0, n * (25 * (sigma * sigma + 0.3)) / p)
        flops += n * (250 + 6 * k) + 30 * pairs
        if backward:
            flops += n * (500 + 20 * k) + 60 * pairs + p * (3 * 11 * 2 * 16 if c["lambda"] > 0 else 10)
    return {"bytes": moved, "flops": flops}


# ---------------------------------------------------------------- the same in 64-bit floats

SSIM_TAPS = (0.00102838, 0.00759876, 0.03600077, 0.10936069, 0.21300554, 0.26601172, 0.21300554, 0.10936069, 0.03600077, 0.00759876,
             0.00102838)


def _sh_basis(d, degree):
    x, y, z = d.unbind(1)
    xx, yy, zz = x * x, y * y, z * z
    b = [torch.full_like(x, 0.28209479177387814)]
    if degree > 0:
        b += [-0.4886025119029199 * y, 0.4886025119029199 * z, -0.4886025119029199 * x]
    if degree > 1:
        b += [1.0925484305920792 * x * y, -1.0925484305920792 * y * z, 0.31539156525252005 * (2 * zz - xx - yy),
              -1.0925484305920792 * x * z, 0.5462742152960396 * (xx - yy)]
    if degree > 2:
        b += [-0.5900435899266435 * y * (3 * xx - yy), 2.890611442640554 * x * y * z, -0.4570457994644658 * y * (4 * zz - xx - yy),
              0.3731763325901154 * z * (2 * zz - 3 * xx - 3 * yy), -0.4570457994644658 * x * (4 * zz - xx - yy),
              1.445305721320277 * z * (xx - yy), -0.5900435899266435 * x * (xx - 3 * yy)]
    return torch.stack(b, 1)


def _project(case, camera, params):
    """The splats in view, front to back: (centre, conic, opacity, colour) with their graph, and extent, radius without."""
    positions, scales, rotations, opacities, sh = params
    V = torch.as_tensor(np.asarray(camera.view), dtype=torch.float64, device=positions.device)
    eye = torch.as_tensor(np.asarray(camera.position), dtype=torch.float64, device=positions.device)
    near = float(np.float32(0.01))
    with torch.no_grad():
        # The order is by depth as single precision has it: world to camera, x, y, z fused in turn.
        z = V[2, 3]
        for a in range(3):
            z = (positions[:, a] * V[2, a] + z).float().double()
    t = positions @ V[:3, :3].T + V[:3, 3]
    tz = t[:, 2]
    o = torch.sigmoid(opacities)
    q = rotations / rotations.norm(dim=1, keepdim=True)
    w, x, y, zq = q.unbind(1)
    R = torch.stack([1 - 2 * (y * y + zq * zq), 2 * (x * y - w * zq), 2 * (x * zq + w * y), 2 * (x * y + w * zq),
                     1 - 2 * (x * x + zq * zq), 2 * (y * zq - w * x), 2 * (x * zq - w * y), 2 * (y * zq + w * x),
                     1 - 2 * (x * x + y * y)], 1).view(-1, 3, 3)
    M = R * torch.exp(scales)[:, None, :]
    lx, ly = 1.3 * 0.5 * camera.width / camera.fx, 1.3 * 0.5 * camera.height / camera.fy
    u, v = (t[:, 0] / tz).clamp(-lx, lx), (t[:, 1] / tz).clamp(-ly, ly)
    zero = torch.zeros_like(tz)
    J = torch.stack([camera.fx / tz, zero, -camera.fx * u / tz, zero, camera.fy / tz, -camera.fy * v / tz], 1).view(-1, 2, 3)
    A = (J @ V[:3, :3]).bmm(M)
    C = A.bmm(A.transpose(1, 2).contiguous())
    dilation = 0.1 if case["mip"] else 0.3
    a, b, cc = C[:, 0, 0] + dilation, C[:, 0, 1], C[:, 1, 1] + dilation
    det = a * cc - b * b
    if case["mip"]:
        raw = C[:, 0, 0] * C[:, 1, 1] - b * b
        o = o * torch.where(raw > 0, raw.clamp(min=1e-300) / det, zero).clamp(min=1e-300).sqrt()
    d = positions - eye
    basis = _sh_basis(d / d.norm(dim=1, keepdim=True), case["degree"])
    colour = (0.5 + (basis[:, :, None] * sh).sum(1)).clamp(min=0)
    centre = torch.stack([camera.fx * t[:, 0] / tz + camera.cx, camera.fy * t[:, 1] / tz + camera.cy], 1)
    conic = torch.stack([cc / det, -b / det, a / det], 1)
    with torch.no_grad():
        mid = 0.5 * (a + cc)
        radius = torch.ceil(3 * torch.sqrt(mid + (mid * mid - det).clamp(min=0.1).sqrt()))
        extent = torch.minimum(torch.stack([a, cc], 1).mul(2 * torch.log(255 * o).clamp(min=0)[:, None]).sqrt(), radius[:, None])
        seen = (z >= near) & (o >= 1 / 255) & (rotations.norm(dim=1) >= 1e-4) & (det > 1e-6)
        seen &= (centre[:, 0] + radius >= 0) & (centre[:, 1] + radius >= 0)
        seen &= (centre[:, 0] - radius <= camera.width) & (centre[:, 1] - radius <= camera.height)
        index = seen.nonzero()[:, 0]
        index = index[torch.sort(z[index], stable=True).indices]
    return centre[index], conic[index], o[index], colour[index], extent[index], radius[index]


class _Raster:
    """Front-to-back blending of the splats over 16x16 tiles, and its derivative; no colour behind."""

    CHUNK, TILES_AT_ONCE = 32, 1024

    def __init__(self, camera, splats):
        self.w, self.h = camera.width, camera.height
        self.centre, self.conic, self.o, self.colour, extent, self.radius = (s.detach() for s in splats)
        device = self.centre.device
        gw, gh = (self.w + 15) // 16, (self.h + 15) // 16
        limit = torch.tensor([gw - 1, gh - 1], device=device)
        low = torch.minimum(((self.centre - extent - 1) / 16).floor().long().clamp(min=0), limit)
        high = torch.minimum(((self.centre + extent + 1) / 16).floor().long().clamp(min=0), limit)
        across = high[:, 0] - low[:, 0] + 1
        count = across * (high[:, 1] - low[:, 1] + 1)
        owner = torch.repeat_interleave(torch.arange(len(count), device=device), count)
        local = torch.arange(len(owner), device=device) - (count.cumsum(0) - count)[owner]
        tile = (low[owner, 1] + local // across[owner]) * gw + low[owner, 0] + local % across[owner]
        tile, order = torch.sort(tile, stable=True)
        self.entries = owner[order]
        sizes = torch.bincount(tile, minlength=gw * gh)
        starts = sizes.cumsum(0) - sizes
        longest = torch.sort(sizes, descending=True).indices
        self.batches = [longest[k:k + self.TILES_AT_ONCE] for k in range(0, gw * gh, self.TILES_AT_ONCE)]
        self.starts, self.sizes = starts, sizes
        p = torch.arange(256, device=device)
        self.px = (torch.arange(gw * gh, device=device) % gw)[:, None] * 16 + (p % 16)
        self.py = (torch.arange(gw * gh, device=device) // gw)[:, None] * 16 + p // 16
        self.inside = (self.px < self.w) & (self.py < self.h)

    def _chunk(self, tiles, at, T, done):
        """The tiles' splats at .. at + CHUNK: indices, offsets, alpha, falloff, transmittance in front of each, taken, and what they leave."""
        k = torch.arange(self.CHUNK, device=tiles.device)
        valid = (at + k)[None, :] < self.sizes[tiles][:, None]
        i = self.entries[torch.where(valid, self.starts[tiles][:, None] + at + k, 0)]
        dx = self.px[tiles][:, None, :] + 0.5 - self.centre[i, 0][..., None]
        dy = self.py[tiles][:, None, :] + 0.5 - self.centre[i, 1][..., None]
        q = self.conic[i]
        power = -0.5 * (q[..., 0, None] * dx * dx + q[..., 2, None] * dy * dy) - q[..., 1, None] * dx * dy
        e = torch.exp(power)
        alpha = (self.o[i][..., None] * e).clamp(max=0.99)
        r = self.radius[i][..., None]
        ok = valid[..., None] & (power <= 0) & (alpha >= 1 / 255) & (dx.abs() <= r) & (dy.abs() <= r)
        keep = torch.where(ok, 1 - alpha, 1.0)
        after = T[:, None, :] * keep.cumprod(1)
        stopped = done[:, None, :] | ((ok & (after < 1e-4)).cumsum(1) > 0)
        taken = ok & ~stopped
        keep = torch.where(taken, keep, 1.0)
        product = keep.cumprod(1)
        front = T[:, None, :] * product / keep
        return i, dx, dy, alpha, e, front, taken, T * product[:, -1], stopped[:, -1]

    def forward(self):
        """The image [h, w, 4]: colour, and the log of the transmittance."""
        device = self.centre.device
        image = torch.zeros(self.h * self.w, 4, dtype=torch.float64, device=device)
        self.fronts = []
        for tiles in self.batches:
            T = torch.ones(len(tiles), 256, dtype=torch.float64, device=device)
            done = ~self.inside[tiles]
            colour = torch.zeros(len(tiles), 256, 3, dtype=torch.float64, device=device)
            states, at, most = [], 0, int(self.sizes[tiles].max())
            while at < most and not bool(done.all()):
                states.append((at, T, done))
                i, _, _, alpha, _, front, taken, T, done = self._chunk(tiles, at, T, done)
                weight = torch.where(taken, front * alpha, 0.0)
                colour = colour + weight.transpose(1, 2).contiguous().bmm(self.colour[i])
                at += self.CHUNK
            self.fronts.append(states)
            inside = self.inside[tiles]
            pixel = (self.py[tiles] * self.w + self.px[tiles])[inside]
            image[pixel] = torch.cat([colour, T.log()[..., None]], 2)[inside]
        return image.view(self.h, self.w, 4)

    def backward(self, adjoint):
        """dL/d(centre, conic, opacity, colour) for dL/dcolour [h, w, 3]."""
        grads = [torch.zeros_like(t) for t in (self.centre, self.conic, self.o, self.colour)]
        adjoint = adjoint.reshape(-1, 3)
        for tiles, states in zip(self.batches, self.fronts):
            inside = self.inside[tiles]
            pixel = torch.where(inside, self.py[tiles] * self.w + self.px[tiles], 0)
            adj = torch.where(inside[..., None], adjoint[pixel], 0.0)
            behind = torch.zeros(inside.shape, dtype=torch.float64, device=adj.device)
            for at, T, done in reversed(states):
                i, dx, dy, alpha, e, front, taken, _, _ = self._chunk(tiles, at, T, done)
                weight = torch.where(taken, front * alpha, 0.0)
                toward = self.colour[i].bmm(adj.transpose(1, 2).contiguous())
                part = weight * toward
                total = part.sum(1)
                after = behind[:, None, :] + total[:, None, :] - part.cumsum(1)
                behind = behind + total
                free = taken & (self.o[i][..., None] * e < 0.99)
                d_alpha = torch.where(free, front * toward - after / (1 - alpha), 0.0)
                d_power = d_alpha * alpha
                q = self.conic[i][..., None]
                at_i = i.reshape(-1)
                grads[0].index_add_(0, at_i, torch.stack([(d_power * (q[:, :, 0] * dx + q[:, :, 1] * dy)).sum(2),
                                                          (d_power * (q[:, :, 1] * dx + q[:, :, 2] * dy)).sum(2)], 2).view(-1, 2))
                grads[1].index_add_(0, at_i, torch.stack([(-0.5 * d_power * dx * dx).sum(2), (-d_power * dx * dy).sum(2),
                                                          (-0.5 * d_power * dy * dy).sum(2)], 2).view(-1, 3))
                grads[2].index_add_(0, at_i, (d_alpha * e).sum(2).view(-1))
                grads[3].index_add_(0, at_i, weight.bmm(adj).view(-1, 3))
        return grads


def _window(x, taps):
    """The 11-tap window both ways over [planes, h, w], cut and renormalised at the border."""
    def pass_over(v):
        k = taps.view(1, 1, 11)
        p, h, w = v.shape
        f = torch.nn.functional.conv1d(v.reshape(p * h, 1, w), k, padding=5).view(p, h, w)
        return f / torch.nn.functional.conv1d(torch.ones(1, 1, w, dtype=v.dtype, device=v.device), k, padding=5).view(1, 1, w)
    return pass_over(pass_over(x).transpose(1, 2).contiguous()).transpose(1, 2)


def _loss(image, target, lam):
    """loss, l1 and ssim of a colour image [h, w, 3] against RGBA8."""
    y = torch.as_tensor(target[..., :3].astype(np.float64) / 255, device=image.device)
    l1 = (image - y).abs().mean()
    taps = torch.tensor(SSIM_TAPS, dtype=torch.float64, device=image.device)
    a, b = image.permute(2, 0, 1), y.permute(2, 0, 1)
    ma, mb = _window(a, taps), _window(b, taps)
    va, vb, cov = _window(a * a, taps) - ma * ma, _window(b * b, taps) - mb * mb, _window(a * b, taps) - ma * mb
    ssim = ((2 * ma * mb + 1e-4) * (2 * cov + 9e-4) / ((ma * ma + mb * mb + 1e-4) * (va + vb + 9e-4))).mean()
    return (1 - lam) * l1 + lam * (1 - ssim), l1, ssim


def exact(case, seed):
    c = {**DEFAULTS, **case}
    if sum(cam.width * cam.height for cam in _cameras(c)) * (8 if c["scene"] == "heavy" else 1) > 2_500_000:
        return None  # half a minute and more
    params = [a.double().requires_grad_() for a in _cloud_arrays(c, seed)]
    n = c["n"]
    stats, total = [], [torch.zeros_like(p) for p in params]
    for k, camera in enumerate(_cameras(c)):
        backward = c["call"] not in ("render", "noalloc")
        with torch.set_grad_enabled(backward):
            splats = _project(c, camera, params)
        raster = _Raster(camera, splats)
        image = raster.forward()
        if not backward:
            return image.view(-1, 4).cpu().numpy() if c["call"] == "render" else image
        colour = image[..., :3].clone().requires_grad_()
        loss, l1, ssim = _loss(colour, _target(camera, seed * 64 + k), c["lambda"])
        stats.append({"loss": loss.item(), "l1": l1.item(), "ssim": ssim.item(), "visible": None})
        adjoint, = torch.autograd.grad(loss, colour)
        for t, g in zip(total, torch.autograd.grad(splats[:4], params, raster.backward(adjoint))):
            t += g
        if c["penalties"] > 0:  # each view's objective has them
            with torch.no_grad():
                s = torch.sigmoid(params[3])
                total[1] += c["penalties"] / n * params[1].exp()
                total[3] += c["penalties"] / n * s * (1 - s)
    if c["call"] in ("gradients", "accumulate"):
        names = ("positions", "scales", "rotations", "opacities", "sh")
        return {"stats": stats[0] if c["call"] == "gradients" else stats, "gradients": {a: t.cpu().numpy() for a, t in zip(names, total)}}
    # Adam's first step moves each parameter with a gradient by its rate against the gradient's sign;
    # the SH values are rounded at random to their storage and have no such value.
    rates = (RATES.position, RATES.scale, RATES.rotation, RATES.opacity)
    moved = {a: (p - rate * torch.sign(g)).detach() for a, p, rate, g in
             zip(("positions", "scales", "rotations", "opacities"), params, rates, total)}
    moved.update({"sh": None} if c["bf16"] else {"sh_dc": None, "sh_rest": None} if c["degree"] > 0 else {"sh_dc": None})
    return {"parameters": moved} if c["call"] in ("queue", "captured") else {"stats": stats[0], "parameters": moved}
