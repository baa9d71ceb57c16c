"""The work a user of this framework has it do, as timed cases.

listed() holds the cases, draw() gives more of the same ranges, prepare() makes what a
program has in hand before the call (sources on the GPU, the visualization with its
steering state, images, training crops), run() makes one pass through the public entry
points and returns its outputs.

  frame      one visualization step of one rank: buffer update (sources, particle cells,
             classification or bricks) and the draw callback, waited for, because the
             simulation overwrites its fields next
  batch      many sub-volumes x camera views in one graph-replayed batch
  train      one step of the occlusion network's training loop: a frame with the plain
             pass, crops of it, one Adam step, the updated parameters
  loss_grad  the network's loss and gradient on given features and targets
  jpeg       the video frame message of a frame in device memory
  composite  sort-last compositing of the sub-volume images one GPU rendered
"""
from __future__ import annotations

import math

import numpy as np
import torch

from isaac_amd import aonet, batch, composite, frame, scenes
from isaac_amd import visualization as V

F16, BF16, F32 = 1, 2, 0


# --------------------------------------------------------------------------- the cases
def _frame(name, scene, size, fb, **kw):
    case = {"kind": "frame", "scene": scene, "x": size[0], "y": size[1], "z": size[2], "w": fb[0], "h": fb[1],
            "particles": 0, "linear": True, "step": 0.5, "dither": 1, "mode": 0, "bricks": False, "dtype": F32,
            "learned": False, "out": "device", "deg": 0.0, "distance": -4.5}
    if name:
        case = {"name": name, **case}
    case.update(kw)
    return case


def listed():
    return [
        # a small run watched while it starts: one scalar field, small window, every launch counts
        _frame("frame_small", "gauss", (64, 64, 64), (512, 512)),
        # the production step: density + vector field + 2 M particles, iso-surface, clipping plane,
        # ambient occlusion, at the camera a session starts with (the volume covers the middle of the frame)
        _frame("frame_production", "prod", (256, 256, 256), (1920, 1080), particles=2_000_000),
        # the same step with the camera moved in until the volume fills the frame
        _frame("frame_production_fill", "prod", (256, 256, 256), (1920, 1080), particles=2_000_000, deg=30.0,
               distance=-2.5),
        # a rank whose box has odd sides, in a window of odd size, with the library's default nearest
        # sampler, a copied (non-persistent) source, functor chains with parameters, particles with
        # radii of their own and blue-noise dithering; the frame goes to host memory, as for IceT
        _frame("frame_ragged_host", "mixed", (181, 127, 203), (1283, 719), particles=150_001, linear=False, dither=3,
               mode=1, out="host", deg=140.0, distance=-3.1),
        # a vector field shown by advected noise (line-integral look), next to a density
        _frame("frame_advection", "field", (192, 192, 192), (1280, 720), deg=75.0, distance=-3.3),
        # a large single field on a 4K wall with fine steps
        _frame("frame_4k", "gauss", (512, 512, 512), (3840, 2160), step=0.25),
        # the precision form with half-precision bricks and the learned occlusion pass
        _frame("frame_bricks_learned", "prod", (256, 256, 256), (1920, 1080), particles=2_000_000, bricks=True,
               dtype=F16, learned=True),
        # many small sub-volumes x views (parameter studies, previews), replayed from one graph
        {"name": "batch_views", "kind": "batch", "volumes": 12, "views": 4, "w": 960, "h": 540, "dtype": F16},
        # training of the occlusion network on the GPU, as aonet.train does it
        {"name": "train_step", "kind": "train", "n": 128, "w": 1920, "h": 1080, "crops": 16, "side": 128},
        # loss and gradient for a program with its own optimiser or data
        {"name": "loss_grad", "kind": "loss_grad", "images": 8, "h": 128, "w": 128},
        # the video frame sent to the server after each step
        {"name": "jpeg_1080p", "kind": "jpeg", "w": 1920, "h": 1080, "quality": 90},
        # eight sub-volume images of one GPU blended in camera order
        {"name": "composite_8", "kind": "composite", "images": 8, "w": 1920, "h": 1080},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame"] * 6 + ["batch", "train", "loss_grad", "jpeg", "composite"])
    fb = (_log(rng, 320, 2560), _log(rng, 240, 1440))
    if kind == "batch":
        return {"kind": "batch", "volumes": rng.randint(2, 12), "views": rng.randint(1, 4),
                "w": rng.randint(240, 960), "h": rng.randint(160, 540), "dtype": rng.choice([F16, BF16, F32])}
    if kind == "train":
        return {"kind": "train", "n": rng.randint(48, 160), "w": max(fb[0], 640), "h": max(fb[1], 480),
                "crops": rng.randint(2, 16), "side": 8 * rng.randint(4, 16)}
    if kind == "loss_grad":
        return {"kind": "loss_grad", "images": rng.randint(1, 8), "h": 8 * rng.randint(4, 24), "w": 8 * rng.randint(4, 24)}
    if kind == "jpeg":
        return {"kind": "jpeg", "w": fb[0], "h": fb[1], "quality": rng.randint(40, 97)}
    if kind == "composite":
        return {"kind": "composite", "images": rng.randint(2, 16), "w": fb[0], "h": fb[1]}
    scene = rng.choice(["gauss", "prod", "prod", "mixed", "field"])
    size = tuple(_log(rng, 48, 288) for _ in range(3))
    if rng.random() < 0.4:  # simulation grids are often cubes with sides of a multiple of 16
        size = (max(48, size[0] // 16 * 16),) * 3
    bricks = scene in ("gauss", "prod") and rng.random() < 0.3
    return _frame(None, scene, size, fb, particles=_log(rng, 2_000, 3_000_000) if scene in ("prod", "mixed") else 0,
                  linear=rng.random() < 0.8, step=rng.choice([0.25, 0.5, 0.5, 0.5, 0.9]), dither=rng.choice([0, 1, 1, 2, 3, 4]),
                  # modes 3 and 4 show surfaces, which the single field without an iso-surface has none of
                  mode=0 if scene == "gauss" else rng.choice([0, 0, 0, 1, 3, 4]), bricks=bricks, dtype=rng.choice([F32, F16, BF16]) if bricks else F32,
                  learned=scene == "prod" and rng.random() < 0.25, out=rng.choice(["device", "device", "host"]),
                  deg=rng.uniform(0.0, 360.0), distance=-rng.uniform(2.3, 4.6))


# --------------------------------------------------------------------------- inputs
def _gaussians(size, rng, dev, count=8):
    """Sum of Gaussians (x fastest: shape Z, Y, X), highest value 1."""
    x, y, z = size
    s = min(size) / 64.0
    out = torch.zeros((z, y, x), device=dev)
    for _ in range(count):
        c = rng.uniform(0.0, 1.0, 3) * np.array(size)
        sig, amp = float(rng.uniform(4.0, 12.0)) * s, float(rng.uniform(0.2, 1.0))
        g = [torch.exp(-((torch.arange(n, device=dev, dtype=torch.float32) + 0.5 - float(c[d])) ** 2) / (2.0 * sig * sig))
             for d, n in enumerate((x, y, z))]
        out += amp * g[2][:, None, None] * g[1][None, :, None] * g[0][None, None, :]
    return out / out.max()


def _noise(size, rng, dev, freq=4, octaves=3):
    """Octaves of interpolated lattice noise in [0, 1]."""
    x, y, z = size
    out = torch.zeros((z, y, x), device=dev)
    for o in range(octaves):
        f = freq * 2 ** o
        lat = torch.from_numpy(rng.uniform(0.0, 1.0, (1, 1, f + 1, f + 1, f + 1)).astype(np.float32)).to(dev)
        out += torch.nn.functional.interpolate(lat, size=(z, y, x), mode="trilinear", align_corners=True)[0, 0] * 0.5 ** o
    out -= out.min()
    return out / out.max()


def _vectors(size, rng, dev):
    """Curl of a noise potential, longest vector 1: (Z, Y, X, 3)."""
    a = [_noise(size, rng, dev, 4, 2) for _ in range(3)]
    d = [torch.gradient(p) for p in a]  # each along z, y, x
    v = torch.stack([d[2][1] - d[1][0], d[0][0] - d[2][2], d[1][2] - d[0][1]], dim=-1)
    return (v / v.square().sum(-1).max().sqrt()).contiguous()


def _particles(n, size, seed, dev):
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    hi = torch.tensor([np.nextafter(np.float32(s), np.float32(0)) for s in size], device=dev)
    pos = torch.minimum(torch.rand((n, 3), generator=g, device=dev) * torch.tensor(size, device=dev, dtype=torch.float32), hi)
    return pos.contiguous(), torch.rand((n, 1), generator=g, device=dev), torch.rand(n, generator=g, device=dev) * 0.6 + 0.2


def _network(seed):
    """Parameters whose output is spread over the occlusion term's range, as a trained network's is."""
    p = aonet.init_params(seed)
    p[-17:-1] *= 0.15
    p[-1] = 0.3
    return p


def _visualization(c, seed):
    dev = torch.device("cuda")
    rng = np.random.default_rng(seed)
    size, fb, scene = (c["x"], c["y"], c["z"]), (c["w"], c["h"]), c["scene"]
    dens = _gaussians(size, rng, dev)
    vols, fields, parts, chains, tfs, iso = [], [], [], [], [], []
    if scene == "gauss":
        vols = [V.VolumeSource("gaussians", dens)]
        chains, tfs, iso = ["idem"], [scenes.SMALL_TF], [0.0]
    elif scene == "prod":
        dens = torch.clamp(0.75 * dens + 0.3 * _noise(size, rng, dev), 0.0, 1.0)
        vols = [V.VolumeSource("density", dens), V.VolumeSource("vector", _vectors(size, rng, dev))]
        chains, tfs, iso = ["idem", "length"], [scenes.DENSITY_TF, scenes.VECTOR_TF], [0.5, 0.0]
    elif scene == "mixed":
        vols = [V.VolumeSource("density", dens, persistent=False), V.VolumeSource("vector", _vectors(size, rng, dev))]
        chains = ["mul(0.9) | add(0.04)", "length | mul(0.8)"]
        tfs, iso = [scenes.DENSITY_TF, scenes.VECTOR_TF], [0.45, 0.0]
    else:
        vols = [V.VolumeSource("density", dens)]
        fields = [V.VolumeSource("flow", _vectors(size, rng, dev))]
        chains, tfs, iso = ["idem", "length"], [scenes.DENSITY_TF, scenes.VECTOR_TF], [0.5, 0.0]
    if c["particles"]:
        pos, attr, radius = _particles(c["particles"], size, seed + 7, dev)
        parts = [V.ParticleSource("particles", pos, attr, radius if scene == "mixed" else None, 0.5)]
        chains, tfs, iso = chains + ["idem"], tfs + [scenes.PARTICLE_TF], iso + [0.0]
    vis = V.IsaacVisualization("perf", fb, size, size, tuple(max(1, s // 4) for s in size), (0, 0, 0), vols, fields, parts)
    vis.functions = chains
    vis.update_functions()
    for i, tf in enumerate(tfs):
        vis.set_transfer_points(i, tf)
    vis.update_transfer()
    vis.iso_threshold = iso
    vis.step, vis.interpolation, vis.dither_mode, vis.render_mode = c["step"], c["linear"], c["dither"], c["mode"]
    if scene != "gauss":
        vis.ambient_occlusion = {"isEnabled": True, "weight": 0.5}
        vis.add_clipping(0.0, 0.0, 0.0, 1.0, 0.0, 0.0)
    vis.background_color = [0.0, 0.0, 0.0, 0.0]
    vis.set_rotation_absolute(scenes.rotation_axis((1.0, 1.0, 0.0), c["deg"]))
    vis.set_distance(c["distance"])
    if c["bricks"]:
        vis.set_render_form(vis.FORM_BRICKS, c["dtype"])
    if c["learned"]:
        vis.aonet_set_params(_network(seed))
        vis.set_ao_mode(vis.AO_LEARNED)
    return vis


def _surface_image(w, h, rng, dev, cover=0.6):
    """A rendered-looking frame: shaded smooth surfaces with fine texture over black, (H, W, 4) uint8."""
    def plane(f):
        lat = torch.from_numpy(rng.uniform(0.0, 1.0, (1, 3, f + 1, f + 1)).astype(np.float32)).to(dev)
        return torch.nn.functional.interpolate(lat, size=(h, w), mode="bicubic", align_corners=True)[0]
    rgb = 0.6 * plane(6) + 0.25 * plane(40) + 0.1 * plane(200)
    level = plane(5)[0]
    mask = level > torch.quantile(level[::8, ::8].reshape(-1), 1.0 - cover)
    img = torch.cat([rgb * mask, mask[None].float()]).clamp(0.0, 1.0)
    return (img * 255.0).to(torch.uint8).permute(1, 2, 0).contiguous()


class _State:
    """What the program holds between passes."""


def prepare(case, seed):
    s = _State()
    s.case = case
    dev = torch.device("cuda")
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "frame":
        s.vis = _visualization(case, seed)
        shape = (case["h"], case["w"], 4)
        s.out = (torch.empty(shape, dtype=torch.uint8, device=dev) if case["out"] == "device"
                 else torch.empty(shape, dtype=torch.uint8, pin_memory=True))
    elif kind == "batch":
        vises, _ = batch.make_subvolumes(0, case["volumes"], seed, (case["w"], case["h"]), case["dtype"],
                                         sides=[batch.SIDES[i % len(batch.SIDES)] for i in range(case["volumes"])])
        s.batch = batch.Batch(vises, case["w"], case["h"])
        s.batch.set_views(*batch.views_for(vises, case["views"], seed))
    elif kind == "train":
        n = case["n"]
        s.vis = _visualization(_frame(None, "prod", (n, n, n), (case["w"], case["h"]), particles=250_000, deg=float(rng.uniform(0, 360)),
                                      distance=-3.0), seed)
        s.vis.aonet_set_params(aonet.init_params(seed))
        s.xy = np.stack([rng.integers(0, case["w"] - case["side"] + 1, case["crops"]),
                         rng.integers(0, case["h"] - case["side"] + 1, case["crops"])], axis=1).astype(np.int32)
    elif kind == "loss_grad":
        n, h, w = case["images"], case["h"], case["w"]
        g = _surface_image(w, n * h, rng, dev, 0.7).float().div(255.0).reshape(n, h, w, 4)
        f = torch.zeros((n, h, w, aonet.FEATURES), device=dev)
        f[..., 0] = (1.0 + g[..., 0]) * g[..., 3]
        f[..., 1] = 1.0 - g[..., 3]
        f[..., 2:5] = torch.nn.functional.normalize(g[..., :3] - 0.5, dim=-1) * g[..., 3:]
        # features a half-precision network input represents exactly
        s.features = f.half().float().cpu().numpy()
        s.target = (g[..., 1] * g[..., 3]).clamp(0.0, 1.0).cpu().numpy()
        s.vis = V.IsaacVisualization("perf", (64, 64), (8, 8, 8), (8, 8, 8), (1, 1, 1), (0, 0, 0), [], [], [])
        s.params = _half_weights(aonet.init_params(seed))
        s.vis.aonet_set_params(s.params)
    elif kind == "jpeg":
        s.rgba = _surface_image(case["w"], case["h"], rng, dev)
        # the send buffer the message is written into (the message of a frame is shorter than its pixels)
        s.send = np.zeros(4 * case["w"] * case["h"] + 4096, np.uint8)
    else:
        s.images = [_surface_image(case["w"], case["h"], rng, dev, 0.35) for _ in range(case["images"])]
        for t in s.images:  # premultiplied colours below full opacity, as the draw callback leaves them
            a = (torch.from_numpy(rng.uniform(0.3, 1.0, 1).astype(np.float32)).to(dev) * t.float()).to(torch.uint8)
            t.copy_(a)
        side = max(1, math.ceil(case["images"] ** (1 / 3)))
        s.positions = [((i % side) * 64, (i // side % side) * 64, (i // side ** 2) * 64) for i in range(case["images"])]
        s.global_size = (64 * side,) * 3
        s.modelview = V.modelview(np.zeros(3), scenes.rotation_axis((1.0, 1.0, 0.0), float(rng.uniform(0, 360))), -3.0)
        s.out = torch.empty_like(s.images[0])
    torch.cuda.synchronize()
    return s


def _half_weights(p):
    """The parameters with every weight a binary16 value, as the matrix cores take them."""
    return p.astype(np.float16).astype(np.float32)


# --------------------------------------------------------------------------- one pass
def run(s):
    kind = s.case["kind"]
    if kind == "frame":
        s.vis.do_visualization(out=s.out)
        s.vis.synchronize()
        return s.out
    if kind == "batch":
        s.batch.render(batch.GRAPH)
        s.batch.synchronize()
        return _device_images(s.batch)
    if kind == "train":
        v = s.vis
        v.update_buffers()
        v.draw(out=False)
        v.aonet_clear_batch()
        v.aonet_add_crops(s.xy, s.case["side"])
        return {"loss": v.aonet_train_step(1e-3), "params": v.aonet_get_params()}
    if kind == "loss_grad":
        loss, grad = s.vis.aonet_loss_grad(s.features, s.target)
        return {"loss": loss, "grad": grad}
    if kind == "jpeg":
        message = frame.jpeg_frame_message(s.rgba, s.case["quality"])
        s.send[:len(message)] = np.frombuffer(message, np.uint8)
        return {"length": len(message), "buffer": s.send}
    order = composite.composite_order(s.positions, [(64, 64, 64)] * len(s.images), s.global_size, (1.0, 1.0, 1.0), s.modelview)
    return composite.composite(s.images, order, out=s.out)


class _DevicePointer:
    def __init__(self, owner, ptr, shape):
        self.owner = owner  # a tensor made from this keeps it, and so the memory
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "|u1", "data": (ptr, False), "version": 2}


def _device_images(b):
    """The batch's frames where they lie in device memory."""
    ptr, n = b.images_device()
    return torch.as_tensor(_DevicePointer(b, ptr, (n, b.height, b.width, 4)), device="cuda")


# --------------------------------------------------------------------------- work, tolerance, oracle
def _march_samples(size, fb, deg, distance, step):
    """Trilinear samples of all rays through the box, from a coarse grid of rays."""
    # vertical field of view of the default projection: perspective(45 rad) -> |tan| of half of it
    ty = abs(math.tan(22.5))
    tx = ty * fb[0] / fb[1]
    n = 96
    u, v = np.meshgrid((np.arange(n) + 0.5) / n * 2 - 1, (np.arange(n) + 0.5) / n * 2 - 1)
    d = np.stack([u * tx, v * ty, -np.ones_like(u)], -1)
    d /= np.linalg.norm(d, axis=-1, keepdims=True)
    rot = scenes.rotation_axis((1.0, 1.0, 0.0), deg)
    d, o = d @ rot, np.array([0.0, 0.0, -distance]) @ rot
    half = np.array(size) / max(size)
    with np.errstate(divide="ignore", invalid="ignore"):
        t0, t1 = (-half - o) / d, (half - o) / d
    near, far = np.minimum(t0, t1).max(-1), np.maximum(t0, t1).min(-1)
    length = np.maximum(0.0, far - np.maximum(near, 0.0)) * max(size) / 2
    return float(length.mean()) * fb[0] * fb[1] / step


def work(case):
    kind = case["kind"]
    net = aonet.flops_per_frame
    if kind == "frame":
        size, fb, scene = (case["x"], case["y"], case["z"]), (case["w"], case["h"]), case["scene"]
        comps = 1 if scene == "gauss" else 4
        vox = size[0] * size[1] * size[2]
        # the iso-surface, the clipping plane and opaque regions end about half of the rays' paths
        samples = _march_samples(size, fb, case["deg"], case["distance"], case["step"]) * (1.0 if scene == "gauss" else 0.5)
        # sources (and the advection texture's old and new state) in, the frame out; a particle's attribute
        b = 4.0 * comps * vox + (2.0 * vox if scene == "field" else 0.0) + 4.0 * case["particles"] + 4.0 * fb[0] * fb[1]
        # per sample: eight corner weights, 8 multiply-adds per channel, compositing; ~30 per classified voxel
        chans = comps if case["bricks"] else 4
        f = samples * ((16 * chans if case["linear"] else 0) + 40) + 30.0 * vox
        return {"bytes": b, "flops": f + (net(*fb) if case["learned"] else 0.0)}
    if kind == "batch":
        sides = [batch.SIDES[i % len(batch.SIDES)] for i in range(case["volumes"])]
        fb = (case["w"], case["h"])
        samples = sum(_march_samples((n, n, n), fb, 30.0, -3.5, 0.5) for n in sides) * case["views"] * 0.5
        value = 4 if case["dtype"] == F32 else 2
        return {"bytes": sum(4.0 * value * n ** 3 for n in sides) + 4.0 * fb[0] * fb[1] * case["views"] * len(sides),
                "flops": samples * (16 * 4 + 40)}
    if kind == "train":
        px = case["crops"] * case["side"] ** 2
        # forward, backward to the data and backward to the weights
        f = 3.0 * net(case["side"], case["side"]) * case["crops"]
        vox = case["n"] ** 3
        return {"bytes": 16.0 * vox + 4.0 * 250_000 + px * 24.0 + 4.0 * 6 * aonet.param_count(), "flops": f + 30.0 * vox}
    if kind == "loss_grad":
        px = case["images"] * case["h"] * case["w"]
        return {"bytes": 36.0 * px + 8.0 * aonet.param_count(), "flops": 3.0 * net(case["w"], case["h"]) * case["images"]}
    px = float(case["w"] * case["h"])
    if kind == "jpeg":
        return {"bytes": 4.0 * px + 0.25 * px, "flops": 60.0 * px}
    return {"bytes": 4.0 * px * (case["images"] + 1), "flops": 12.0 * px * (case["images"] - 1)}


def tolerance(case):
    kind = case["kind"]
    if kind == "train":
        # Adam's first steps move every parameter by the learning rate times the sign of its
        # gradient, so a gradient near zero that changes sign under another order of sums moves
        # its parameter by two learning rates
        return {"rel": 1e-3, "max": 0.1}
    if kind == "loss_grad":
        # binary16 activations and activation gradients: 4e-4 to 1.5e-3 from the 64-bit gradient
        return {"rel": 5e-3, "max": 0.1}
    if kind == "frame" and case["learned"]:
        # the network's binary16 activations round differently under another order of its
        # sums, and the occlusion term then moves shaded bytes across a rounding boundary (5e-5 of
        # the bytes with every bias moved by 1e-6)
        return {"differ": 0.0002}
    return "exact"


def exact(case, seed):
    """The loss and gradient in 64 bits.  None for the others: frames, messages and composites
    are bytes, and a training step starts from the framework's own rendered frame."""
    if case["kind"] != "loss_grad":
        return None
    s = prepare(case, seed)
    dev = torch.device("cuda")
    p = torch.from_numpy(s.params.astype(np.float64)).to(dev).requires_grad_(True)
    x = torch.from_numpy(s.features.astype(np.float64)).to(dev)
    target = torch.from_numpy(s.target.astype(np.float64)).to(dev)
    weights, at = {}, 0
    for name, ci, co in aonet.LAYERS:
        weights[name] = (p[at:at + co * 9 * ci].reshape(co, 9, ci), p[at + co * 9 * ci:at + co * 9 * ci + co])
        at += co * 9 * ci + co

    def layer(name, t):
        w, b = weights[name]
        n, h, wd, c = t.shape
        padded = torch.nn.functional.pad(t, (0, 0, 1, 1, 1, 1))
        z = b.expand(n, h, wd, -1).reshape(-1, b.numel())
        for tap in range(9):
            ky, kx = divmod(tap, 3)
            z = z + padded[:, ky:ky + h, kx:kx + wd, :].reshape(-1, c) @ w[:, tap, :].t().contiguous()
        return torch.relu(z).reshape(n, h, wd, -1)

    def pool(t):
        n, h, wd, c = t.shape
        return t.reshape(n, h // 2, 2, wd // 2, 2, c).mean(dim=(2, 4))

    def up(t):
        return t.repeat_interleave(2, dim=1).repeat_interleave(2, dim=2)

    s0 = layer("e0b", layer("e0a", x))
    s1 = layer("e1b", layer("e1a", pool(s0)))
    s2 = layer("e2b", layer("e2a", pool(s1)))
    t = layer("e3b", layer("e3a", pool(s2)))
    t = layer("d2", torch.cat([up(t), s2], dim=3))
    t = layer("d1", torch.cat([up(t), s1], dim=3))
    t = layer("d0", torch.cat([up(t), s0], dim=3))
    out = t @ p[at:at + aonet.HEAD_IN] + p[at + aonet.HEAD_IN]
    loss = (out - target).square().sum()
    grad, = torch.autograd.grad(loss, p)
    return {"loss": float(loss), "grad": grad}
