"""The renderer's workloads as timed cases: what a user of the framework has it do.

A case is a dict of plain values; ``prepare`` builds what a program holds before the call
(volumes in memory, poses, a renderer or context, output planes), ``run`` is one pass through
the public entry points, ``work`` the bytes and operations it cannot do without, ``exact``
the same outputs in 64 bits where they have such a value.

Kinds of case:
  view      ``VolumeRenderer.render`` of a resident volume into host arrays: the viewer
  load      ``VolumeRenderer.set_data`` of the next timepoint, then its frame: the time slider
  frame     ``Context.render_slot`` into device planes (max projection, opacity, iso surface)
  batch     ``Context.render_batch``: timepoints x poses of one size, the movie recorder
  serve     ``Context.render_frames``: frames of mixed sizes and settings, the render server
  learned   ``LearnedMIP.render_judged_many``: coarse frames through the network, judged
  train     ``Net.gradients``: the loss and its gradient on one batch of coarse / fine pairs

Volumes are Gaussian blobs over a camera background with shot and read noise, 2000 blobs per
512^3 voxels (the recipe of the repository's synthetic workloads).
"""
import math

import numpy as np
import torch

from spimagine_amd import _lib, learned, synth
from spimagine_amd.utils import mat4_perspective
from spimagine_amd.volumerender import VolumeRenderer
from spimagine_amd.volumerender.volumerender import render_matrices

ITEM = {"f32": 4, "u16": 2, "u8": 1}
NUMPY = {"f32": np.float32, "u16": np.uint16, "u8": np.uint8}


# --------------------------------------------------------------------------------- cases
def _steps(nx, ny, nz):
    """At most one voxel a step, in whole 16-sample blocks."""
    return synth.steps_for_shape((nz, ny, nx))


def listed():
    return [
        # the smallest call: a preview of a small float stack at the widget's default size
        # and the configuration's default step count, latency and host work included
        dict(name="view_small_f32", kind="view", dtype="f32", nx=128, ny=128, nz=128, w=200, h=200,
             steps=200, method="mip", filter="linear", alpha_pow=0., gamma=1., uz=1., pose=1),
        # turning a 512^3 stack in the viewer: default steps, a window that is not square, a
        # stack whose planes lie further apart than its pixels
        dict(name="view_u16_default", kind="view", dtype="u16", nx=512, ny=512, nz=512, w=1000,
             h=700, steps=200, method="mip", filter="linear", alpha_pow=0., gamma=1., uz=1.5, pose=2),
        # the time slider: the next timepoint goes to the device and is drawn
        dict(name="load_u16_timepoint", kind="load", dtype="u16", nx=512, ny=512, nz=256, w=512,
             h=512, steps=200, method="mip", filter="linear", alpha_pow=0., gamma=1., uz=1., pose=3),
        # the headline frame: max projection at one voxel a step
        dict(name="mip_u16_headline", kind="frame", dtype="u16", nx=1024, ny=1024, nz=512, w=1024,
             h=1024, steps=1536, method="mip", filter="linear", alpha_pow=0., gamma=1., uz=1., pose=0),
        # the largest frame: a volume above 4 GiB at 2048^2, the serving workload's tail
        dict(name="mip_u16_wide_2048", kind="frame", dtype="u16", nx=2048, ny=2048, nz=512, w=2048,
             h=2048, steps=_steps(2048, 2048, 512), method="mip", filter="linear", alpha_pow=0.,
             gamma=1., uz=1., pose=4),
        # the opacity transfer mode
        dict(name="opacity_u16_512", kind="frame", dtype="u16", nx=512, ny=512, nz=512, w=1024,
             h=1024, steps=896, method="mip", filter="linear", alpha_pow=.6, gamma=1., uz=1., pose=5),
        # the iso surface with its normal smoothing and occlusion
        dict(name="iso_u16_512", kind="frame", dtype="u16", nx=512, ny=512, nz=512, w=1024, h=1024,
             steps=896, method="iso", filter="linear", alpha_pow=0., gamma=1., uz=1., pose=6),
        # an 8-bit stack of odd sizes with the nearest filter and a gamma
        dict(name="mip_u8_nearest_odd", kind="frame", dtype="u8", nx=511, ny=509, nz=257, w=777,
             h=613, steps=_steps(511, 509, 257), method="mip", filter="nearest", alpha_pow=0.,
             gamma=.7, uz=1., pose=7),
        # a movie over a time lapse: 8 timepoints x 8 poses in one launch
        dict(name="batch_u16_movie", kind="batch", dtype="u16", nx=1024, ny=1024, nz=256, w=1024,
             h=1024, steps=_steps(1024, 1024, 256), times=8, poses=8, filter="linear", alpha_pow=0.,
             gamma=1., pose=8),
        # the render server: whatever is waiting, frames of several sizes, boxes and steps
        dict(name="serve_f32_mixed", kind="serve", dtype="f32", nx=256, ny=256, nz=256, volumes=3,
             frames=12, wmin=256, wmax=1024, steps=_steps(256, 256, 256), filter="linear",
             alpha_pow=0., gamma=1., pose=9),
        # learned frames, each judged against the exact renderer
        dict(name="learned_judged_8", kind="learned", dtype="u16", nx=512, ny=512, nz=512, w=1024,
             h=1024, steps=896, frames=8, pose=10),
        # one training batch of the network (the trainer's own sizes)
        dict(name="train_8x512", kind="train", frames=8, w=512, h=512),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["view", "view", "load", "frame", "frame", "frame", "batch", "serve",
                       "learned", "train"])
    pose = rng.randrange(1 << 20)
    if kind == "train":
        return dict(kind=kind, frames=rng.randint(1, 8), w=4 * rng.randint(16, 128),
                    h=4 * rng.randint(16, 128))
    if kind == "learned":
        n = 2 * rng.randint(96, 256)
        return dict(kind=kind, dtype="u16", nx=n, ny=n, nz=2 * rng.randint(48, n // 2),
                    w=16 * rng.randint(24, 64), h=16 * rng.randint(24, 64), steps=_steps(n, n, n),
                    frames=rng.randint(1, 8), pose=pose)
    dtype = rng.choice(["u16", "u16", "u8", "f32"])
    top = 1024 if kind == "frame" else 512
    nx, ny, nz = _log(rng, 48, top), _log(rng, 48, top), _log(rng, 48, 512)
    c = dict(kind=kind, dtype=dtype, nx=nx, ny=ny, nz=nz,
             steps=rng.choice([200, _steps(nx, ny, nz), 16 * rng.randint(4, 64)]),
             filter=rng.choice(["linear", "linear", "linear", "nearest"]),
             alpha_pow=rng.choice([0., 0., round(rng.uniform(.2, 1.2), 2)]),
             gamma=rng.choice([1., 1., round(rng.uniform(.5, 2.), 2)]), pose=pose)
    if kind in ("view", "load", "frame"):
        c.update(w=_log(rng, 128, 1400), h=_log(rng, 128, 1400),
                 method=rng.choice(["mip", "mip", "mip", "iso"]),
                 uz=rng.choice([1., round(rng.uniform(.5, 4.), 2)]))
        if c["method"] == "iso":
            c["alpha_pow"] = 0.
    elif kind == "batch":
        c.update(w=_log(rng, 128, 1024), h=_log(rng, 128, 1024), times=rng.randint(1, 6),
                 poses=rng.randint(1, 8))
    else:
        c.update(volumes=rng.randint(1, 4), frames=rng.randint(2, 16), wmin=128, wmax=1024)
    return c


# --------------------------------------------------------------------------------- inputs
def _tile(n, count, sigma, rng):
    """(n, n, n) float32 sum of `count` unit-background blobs that wrap around its edges,
    added one by one (the same values in every process)."""
    m = int(math.ceil(3 * sigma[1]))
    tile = torch.zeros((n + 2 * m,) * 3, device="cuda")
    ax = torch.arange(n + 2 * m, device="cuda", dtype=torch.float32)
    centres, sigmas = rng.uniform(m, n + m, (count, 3)), rng.uniform(*sigma, (count, 3))
    amps = rng.uniform(0., 1., count)
    for c, s, a in zip(centres, sigmas, amps):
        lo = [int(max(0, math.floor(x - 3 * y))) for x, y in zip(c, s)]
        hi = [int(min(n + 2 * m, math.ceil(x + 3 * y) + 1)) for x, y in zip(c, s)]
        g = [torch.exp(-.5 * ((ax[p:q] - float(x)) / float(y)) ** 2)
             for p, q, x, y in zip(lo, hi, c, s)]
        tile[lo[0]:hi[0], lo[1]:hi[1], lo[2]:hi[2]] += (
            float(a) * .833 + .167) * g[0][:, None, None] * g[1][None, :, None] * g[2][None, None, :]
    for d in range(3):  # fold the margins over
        tile.narrow(d, n, m).add_(tile.narrow(d, 0, m).clone())
        tile.narrow(d, m, m).add_(tile.narrow(d, n + m, m).clone())
        tile = tile.narrow(d, m, n)
    return tile.contiguous()


def _volume(dtype, nx, ny, nz, seed):
    """A device volume (uint16 as its int16 bit pattern) from the seed alone."""
    rng = np.random.default_rng(seed)
    n = 256 if max(nx, ny, nz) > 160 else 128
    sigma = (3., 10.) if n == 256 else (2., 6.)
    tile = _tile(n, 250 if n == 256 else 40, sigma, rng)
    reps = [-(-k // n) for k in (nz, ny, nx)]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed) + 1)
    out = torch.empty((nz, ny, nx), device="cuda",
                      dtype={"f32": torch.float32, "u16": torch.int16, "u8": torch.uint8}[dtype])
    for k in range(reps[0]):  # one slab of tiles at a time, each tile turned its own way
        rows = []
        for j in range(reps[1]):
            row = []
            for i in range(reps[2]):
                t = torch.flip(tile, [d for d in range(3) if rng.integers(2)])
                row.append(torch.roll(t, [int(v) for v in rng.integers(0, n, 3)], (0, 1, 2)))
            rows.append(torch.cat(row, 2))
        z0, z1 = k * n, min(nz, k * n + n)
        slab = torch.cat(rows, 1)[:z1 - z0, :ny, :nx]
        noise = torch.randn(slab.shape, generator=gen, device="cuda")
        if dtype == "f32":
            out[z0:z1] = slab + .05 + .02 * noise
        elif dtype == "u8":
            out[z0:z1] = (20. + 180. * slab + 3. * noise).round_().clamp_(0, 255).to(torch.uint8)
        else:
            shot = torch.poisson(100. + 3000. * slab, generator=gen)
            v = (shot + 5. * noise).round_().clamp_(0, 65535).to(torch.int32)
            out[z0:z1] = torch.where(v >= 32768, v - 65536, v).to(torch.int16)
    return out


def _trained_like(nx, ny, nz, seed):
    """A volume of the network's training recipe (every blob on its own)."""
    cfg = dict(synth.CONFIGS["iso"], shape=(nz, ny, nx),
               n_blobs=max(8, int(round(2000. * nx * ny * nz / 512 ** 3))))
    return synth.blob_volume_device(seed=seed, **cfg)


def _range(c):
    """The transfer range a user sets: background to bright."""
    return {"f32": (.05, .9), "u16": (100., 2500.), "u8": (20., 200.)}[c["dtype"]]


def _host(vol, dtype):
    return vol.cpu().numpy().view(NUMPY[dtype])


def _pose(c, k=0):
    return synth.random_poses(k + 1, seed=c["pose"])[k] if c["pose"] else synth.headline_camera()[0]


def _projection(c):
    return mat4_perspective(45, 1. * c.get("w", 1) / c.get("h", 1), .1, 10)


def _matrices(c, k=0, projection=None):
    return render_matrices(_pose(c, k), _projection(c) if projection is None else projection,
                           (c["nx"], c["ny"], c["nz"]), (1., 1., c.get("uz", 1.)))


def _params(c, k=0, **more):
    lo, hi = _range(c)
    inv_p, inv_m = _matrices(c, k, more.pop("projection", None))
    lo, hi = more.pop("span", (lo, hi))
    a = dict(box=(-1, 1, -1, 1, -1, 1), min_val=lo, max_val=hi, gamma=c.get("gamma", 1.),
             alpha_pow=c.get("alpha_pow", 0.), max_steps=c["steps"],
             filter=_lib.FILTER_NEAREST if c.get("filter") == "nearest" else _lib.FILTER_LINEAR)
    a.update(more)
    return _lib.make_params(inv_p, inv_m, **a)


def _mixed(c):
    """The frames of a serve case: (volume, width, height, pose index, box, steps)."""
    rng = np.random.default_rng(c["pose"])
    out = []
    for k in range(c["frames"]):
        w, h = np.exp(rng.uniform(np.log(c["wmin"]), np.log(c["wmax"]), 2)).astype(int)
        box = (-1., 1., -1., 1., -1., 1.) if rng.integers(3) else (-1., 1., -.5, 1., -1., .6)
        steps = c["steps"] if rng.integers(3) else max(16, c["steps"] // 2)
        out.append((int(rng.integers(c["volumes"])), int(w), int(h), k, box, steps))
    return out


def _renderer(c):
    r = VolumeRenderer((c["w"], c["h"]), interpolation=c["filter"])
    lo, hi = _range(c)
    r.set_max_steps(c["steps"])
    r.set_min_val(lo)
    r.set_max_val(hi)
    r.set_gamma(c["gamma"])
    r.set_alpha_pow(c["alpha_pow"])
    r.set_units([1., 1., c["uz"]])
    r.set_projection(_projection(c))
    r.set_modelView(_pose(c))
    return r


def _add(ctx, vol, dtype):
    return ctx.volume_add(dev_ptr=vol.data_ptr(), dtype=NUMPY[dtype], shape=tuple(vol.shape))


def prepare(c, seed):
    kind = c["kind"]
    if kind == "train":
        gen = torch.Generator(device="cuda")
        gen.manual_seed(int(seed))
        n, h, w = c["frames"], c["h"], c["w"]
        fine = _frames_like(n, 2 * h, 2 * w, gen)
        coarse = torch.nn.functional.avg_pool2d(fine, 2)
        planes = torch.cat([coarse, torch.nn.functional.max_pool2d(fine, 2)], 1).contiguous()
        params, _ = learned.load_weights(learned.WEIGHTS_PATH)
        return dict(c=c, planes=planes, target=fine[:, 0].contiguous(), params=params,
                    net=learned.Net(0, params), stream=torch.cuda.Stream())
    if kind in ("view", "load"):
        vol = _host(_volume(c["dtype"], c["nx"], c["ny"], c["nz"], seed), c["dtype"])
        r = _renderer(c)
        r.set_data(vol)
        return dict(c=c, vol=vol, rend=r)
    ctx = _lib.Context(0)
    count = c.get("times", c.get("volumes", 1))
    slots = []
    for k in range(count):
        vol = (_trained_like(c["nx"], c["ny"], c["nz"], seed) if kind == "learned" else
               _volume(c["dtype"], c["nx"], c["ny"], c["nz"], seed + 1000 * k))
        slots.append(_add(ctx, vol, c["dtype"]))
    s = dict(c=c, ctx=ctx, slots=slots, stream=torch.cuda.Stream())
    if kind == "frame":
        planes = [torch.zeros((c["h"], c["w"]), device="cuda") for _ in range(4)]
        s.update(params=_params(c), planes=planes,
                 normals=torch.zeros((c["h"], c["w"], 3), device="cuda"))
    elif kind == "batch":
        n = c["times"] * c["poses"]
        s["out"] = torch.zeros((n, 2, c["h"], c["w"]), device="cuda")
        ms = [_matrices(c, k) for k in range(c["poses"])]
        at = s["out"].data_ptr() + 8 * c["w"] * c["h"] * np.arange(n, dtype=np.uint64)
        s["jobs"] = _lib.jobs_from_arrays(
            [slots[k // c["poses"]] for k in range(n)], [ms[k % c["poses"]][0] for k in range(n)],
            [ms[k % c["poses"]][1] for k in range(n)], at, at + 4 * c["w"] * c["h"])
        s["params"] = _params(c)
    elif kind == "serve":
        s["outs"], s["frames"] = [], []
        for v, w, h, k, box, steps in _mixed(c):
            o = torch.zeros((2, h, w), device="cuda")
            p = _params(c, k, projection=mat4_perspective(45, 1. * w / h, .1, 10), box=box,
                        max_steps=steps)
            s["outs"].append(o)
            s["frames"].append(_lib.make_frame(slots[v], p, w, h, o[0].data_ptr(), o[1].data_ptr()))
    elif kind == "learned":
        s["lm"] = learned.LearnedMIP(ctx)
        s["lm"].attach(slots[0])
        # the network's frames are trained on each volume's own range
        span = [float(v) for v in torch.aminmax(_float(vol, c["dtype"]))]
        s["params"] = [_params(c, k, span=span) for k in range(c["frames"])]
        s["out"] = torch.zeros((2, c["frames"], c["h"], c["w"]), device="cuda")
    return s


def _frames_like(n, h, w, gen):
    """(n, 1, h, w) images of soft spots in [0, 1], as max projections look."""
    x = torch.rand((n, 1, -(-h // 16), -(-w // 16)), generator=gen, device="cuda") ** 4
    x = torch.nn.functional.interpolate(x, scale_factor=16, mode="bilinear")[:, :, :h, :w]
    return (x + .02 * torch.rand(x.shape, generator=gen, device="cuda")).clamp(0, 1)


# --------------------------------------------------------------------------------- a pass
def run(s):
    c = s["c"]
    kind = c["kind"]
    if kind in ("view", "load"):
        r = s["rend"]
        if kind == "load":
            r.set_data(s["vol"])
        if c["method"] == "iso":
            r.render(method="iso_surface")
            return [r.output, r.output_alpha, r.output_depth, r.output_normals, r.output_occlusion]
        r.render()
        return [r.output, r.output_alpha]
    st = s["stream"].cuda_stream
    if kind == "train":
        n, _, h, w = s["planes"].shape
        grad, sse = s["net"].gradients(s["planes"].data_ptr(), s["target"].data_ptr(), n, h, w, st)
        return [grad, sse]
    ctx = s["ctx"]
    if kind == "frame":
        p, (out, alpha, depth, occ) = s["params"], s["planes"]
        if c["method"] == "iso":
            ctx.render_slot(s["slots"][0], p, _lib.METHOD_ISO_SURFACE, c["w"], c["h"],
                            out.data_ptr(), alpha.data_ptr(), depth.data_ptr(),
                            s["normals"].data_ptr(), occ.data_ptr(), stream=st)
            return [out, alpha, depth, s["normals"], occ]
        ctx.render_slot(s["slots"][0], p, _lib.METHOD_MAX_PROJECT, c["w"], c["h"], out.data_ptr(),
                        alpha.data_ptr(), stream=st)
        return [out, alpha]
    if kind == "batch":
        ctx.render_batch(s["jobs"], c["w"], c["h"], stream=st, params=s["params"])
        return [s["out"]]
    if kind == "serve":
        nearest = c["filter"] == "nearest"
        ctx.render_frames(s["frames"], alpha_pow=c["alpha_pow"], stream=st,
                          filter=_lib.FILTER_NEAREST if nearest else _lib.FILTER_LINEAR)
        return s["outs"]
    out, alpha = s["out"]
    s["lm"].render_judged_many(s["slots"][0], s["params"], list(out), list(alpha), s["stream"],
                               wait=False)
    return [out, alpha]


# ----------------------------------------------------------------------- in 64 bits, and work
def _rays(inv_p, inv_m, w, h, box, device):
    """Origin, direction (texture units are (1 + x) / 2), entry and exit of every pixel's ray."""
    f = dict(dtype=torch.float64, device=device)
    u = torch.arange(w, **f) / w * 2 - 1
    v = torch.arange(h, **f) / h * 2 - 1
    v, u = torch.meshgrid(v, u, indexing="ij")
    P = torch.tensor(np.asarray(inv_p, np.float64).reshape(4, 4), device=device)
    M = torch.tensor(np.asarray(inv_m, np.float64).reshape(4, 4), device=device)
    one = torch.ones_like(u)
    front = torch.stack([u, v, -one, one], -1) @ P.T
    back = torch.stack([u, v, one, one], -1) @ P.T
    front, back = front / front[..., 3:], back / back[..., 3:]
    o = front @ M.T
    o = o / o[..., 3:]
    d = back - front
    d = (d / d.norm(dim=-1, keepdim=True)) @ M.T
    o, d = o[..., :3], d[..., :3]
    b = torch.tensor(np.asarray(box, np.float64).reshape(3, 2), device=device)
    t0, t1 = (b[:, 0] - o) / d, (b[:, 1] - o) / d
    near, far = torch.minimum(t0, t1).amax(-1), torch.maximum(t0, t1).amin(-1)
    return o, d, near, far


def _exact_frame(c, vol, p, w, h):
    """[output, alpha] of a max or opacity projection; vol: a float32 device volume."""
    nearest, short = p.filter == _lib.FILTER_NEAREST, c["dtype"] != "f32"
    o, d, near, far = _rays(list(p.inv_p), list(p.inv_m), w, h, list(p.box), vol.device)
    hit = (far > near).reshape(-1)
    o, d = o.reshape(-1, 3)[hit], d.reshape(-1, 3)[hit]
    near, far = near.reshape(-1)[hit].clamp(min=0.), far.reshape(-1)[hit]
    n = (p.max_steps // 16) * 16
    pos = (1. + o + near[:, None] * d) * .5
    step = ((far - near).abs() / n)[:, None] * d * .5
    size = torch.tensor([vol.shape[2], vol.shape[1], vol.shape[0]], device=vol.device)
    flat, sy, sz = vol.view(-1), vol.shape[2], vol.shape[1] * vol.shape[2]
    top = size - 1
    zero = torch.zeros_like(top)
    col = torch.zeros(len(pos), dtype=torch.float64, device=vol.device)
    left, broke = torch.ones_like(col), torch.zeros_like(col, dtype=torch.bool)
    taken = torch.zeros_like(col)
    a = p.alpha_pow ** 2 * (.1 if short else 1.)
    for k in range(n + 16):
        q = (pos + (taken[:, None] if p.alpha_pow else k) * step) * size
        if nearest:
            i = torch.minimum(torch.maximum(q.floor().long(), zero), top)
            v = flat[i[:, 0] + sy * i[:, 1] + sz * i[:, 2]].double()
        else:
            q = q - .5
            f = q.floor()
            t, f = q - f, f.long()
            lo = torch.minimum(torch.maximum(f, zero), top)
            hi = torch.minimum(torch.maximum(f + 1, zero), top)
            z = []
            for iz in (lo[:, 2], hi[:, 2]):
                y = []
                for iy in (lo[:, 1], hi[:, 1]):
                    row = sy * iy + sz * iz
                    x0, x1 = flat[row + lo[:, 0]].double(), flat[row + hi[:, 0]].double()
                    y.append(x0 + t[:, 0] * (x1 - x0))
                z.append(y[0] + t[:, 1] * (y[1] - y[0]))
            v = z[0] + t[:, 2] * (z[1] - z[0])
        if not p.alpha_pow:
            col = torch.maximum(col, v)
            continue
        if k % 16 == 0:  # a ray that ran out of light stops only until its next 16 samples
            broke.zero_()
        v = (v - p.min_val) / (p.max_val - p.min_val)
        col = torch.where(broke, col, torch.maximum(col, left * v))
        left = torch.where(broke, left, left * (1. - a * (v if short else v.clamp(0, 1))))
        taken = torch.where(broke, taken, taken + 1)
        broke |= left <= .01
    if not p.alpha_pow:
        col = (col - p.min_val) / (p.max_val - p.min_val)
    col = col.clamp(min=0.) if p.gamma == 1. else col.clamp(min=0.) ** p.gamma
    out = torch.zeros(w * h, dtype=torch.float64, device=vol.device)
    alpha = torch.full_like(out, 0. if short else -1.)
    out[hit] = col.clamp(0., 1.)
    alpha[hit] = near if short else 1.
    return [out.view(h, w), alpha.view(h, w)]


def _float(vol, dtype):
    return vol if dtype == "f32" else vol.float() if dtype == "u8" else torch.where(
        vol < 0, vol.float() + 65536., vol.float())


def exact(c, seed):
    kind = c["kind"]
    if kind == "learned" or c.get("method") == "iso":
        # a learned frame is kept or replaced by an estimate, an iso pixel is hit or missed
        # by a comparison of rounded samples: no value in 64 bits
        return None
    if kind == "train":
        return _exact_gradient(prepare(c, seed))
    if kind in ("view", "load", "frame"):
        if 1. * c["w"] * c["h"] * c["steps"] > 4e9:
            return None
        vol = _float(_volume(c["dtype"], c["nx"], c["ny"], c["nz"], seed), c["dtype"])
        return _exact_frame(c, vol, _params(c), c["w"], c["h"])
    frames = _mixed(c) if kind == "serve" else []
    samples = (sum(w * h * steps for _, w, h, _, _, steps in frames) if frames
               else c["w"] * c["h"] * c["steps"] * c["times"] * c["poses"])
    if 1. * samples > 6e9:
        return None
    vols = {}

    def vol(k):
        if k not in vols:
            vols[k] = _float(_volume(c["dtype"], c["nx"], c["ny"], c["nz"], seed + 1000 * k),
                             c["dtype"])
        return vols[k]

    if kind == "serve":
        return [torch.stack(_exact_frame(
            c, vol(v), _params(c, k, projection=mat4_perspective(45, 1. * w / h, .1, 10), box=box,
                               max_steps=steps), w, h)) for v, w, h, k, box, steps in frames]
    return [torch.stack([torch.stack(_exact_frame(c, vol(t), _params(c, k), c["w"], c["h"]))
                         for t in range(c["times"]) for k in range(c["poses"])])]


def _exact_gradient(s):
    """The network's gradient and summed squared error in float64 (no bf16 rounding)."""
    n, _, h, w = s["planes"].shape
    ps = {}
    for name, v in learned.split_params(np.asarray(s["params"], np.float64)).items():
        ps[name] = torch.tensor(v, device="cuda", requires_grad=True)

    def conv(x, name):
        pad = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
        y = ps[name + ".b"]
        for t in range(9):
            y = y + pad[:, t // 3:t // 3 + x.shape[1], t % 3:t % 3 + x.shape[2]] @ ps[name + ".w"][t]
        return y

    def pool(x):
        return x.unflatten(2, (-1, 2)).unflatten(1, (-1, 2)).mean((2, 4))

    def up(x):
        return x.repeat_interleave(2, 1).repeat_interleave(2, 2)

    planes = s["planes"].double()
    x = planes.permute(0, 2, 3, 1)
    e0b = conv(conv(conv(x, "in").relu(), "e0").relu(), "e0b").relu()
    e1b = conv(conv(pool(e0b), "e1").relu(), "e1b").relu()
    e2 = conv(conv(pool(e1b), "e2a").relu(), "e2").relu()
    u1 = conv(up(e2) + e1b, "u1").relu()
    u0b = conv(conv(up(u1) + e0b, "u0").relu(), "u0b").relu()
    r = conv(u0b, "head").unflatten(3, (2, 2)).permute(0, 1, 3, 2, 4).reshape(n, 2 * h, 2 * w)
    base = torch.nn.functional.interpolate(planes[:, :1], scale_factor=2, mode="bilinear")[:, 0]
    sse = ((r + base - s["target"].double()) ** 2).sum()
    (sse / (n * 4 * h * w)).backward()
    return [torch.cat([p.grad.reshape(-1) for p in ps.values()]), float(sse)]


def _hit_samples(c, p, w, h):
    _, _, near, far = _rays(list(p.inv_p), list(p.inv_m), w, h, list(p.box), "cpu")
    n = p.max_steps if c.get("method") == "iso" else (p.max_steps // 16 + 1) * 16
    return float((far > near).sum()) * n


def work(c):
    """Volumes read once and outputs written once; one trilinear sample is 14 operations of
    interpolation and 6 of its position, a network pixel 2 x 9 x 32 x 32 a layer."""
    kind = c["kind"]
    if kind == "train":
        px = c["frames"] * c["h"] * c["w"]
        # forward and two backward products of the layers: five and a half at full size (the
        # input and head layers are thin), three at half, two at a quarter
        macs = px * (2 * 9 * 32 + 9 * 32 * 4 + 9 * 32 * 32 * (4 + 3 / 4. + 2 / 16.))
        return {"bytes": 4. * px * 6 + 4. * learned.param_count() * 2, "flops": 6. * macs}
    voxels = 1. * c["nx"] * c["ny"] * c["nz"] * ITEM[c["dtype"]]
    if kind == "serve":
        fs = _mixed(c)
        px = sum(w * h for _, w, h, _, _, _ in fs)
        samples = sum(_hit_samples(c, _params(c, k, projection=mat4_perspective(45, 1. * w / h, .1, 10),
                                              box=box, max_steps=steps), w, h)
                      for _, w, h, k, box, steps in fs)
        vols = len({f[0] for f in fs})
        return {"bytes": vols * voxels + 8. * px, "flops": 20. * samples}
    px = c["w"] * c["h"]
    if kind == "learned":
        # the coarse frames' samples (a quarter of the pixels and of the steps, two channels)
        # and the network; the judge's sparse pixels
        coarse = sum(_hit_samples(c, _params(c, k, max_steps=max(16, c["steps"] // 4)), c["w"] // 2,
                                  c["h"] // 2) for k in range(c["frames"]))
        macs = px / 4. * (2 * 9 * 32 + 9 * 32 * 4 + 9 * 32 * 32 * (4 + 3 / 4. + 2 / 16.))
        return {"bytes": voxels / 4 + 8. * px * c["frames"],
                "flops": 34. * coarse + 2. * macs * c["frames"]}
    poses = c.get("poses", 1)
    times = c.get("times", 1)
    samples = times * sum(_hit_samples(c, _params(c, k), c["w"], c["h"]) for k in range(poses))
    ops = 4. if c["filter"] == "nearest" else 20.
    planes = 28. if c.get("method") == "iso" else 8.
    # a timepoint that is uploaded is read from the host and written to the device as well
    moved = 3. if kind == "load" else 1.
    return {"bytes": moved * times * voxels + planes * px * times * poses, "flops": ops * samples}
