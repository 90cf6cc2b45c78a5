"""GPU: the march that the default tuning picks for a frame or a batch is not slower than the
staged one (a chunk length picks that, SPR_TUNE_CHUNK), on volumes that leave little to skip or
whose bounds promise more than they keep; and the frames are the same, bit for bit."""
import numpy as np
import pytest

from spimagine_amd import _lib
from spimagine_amd.utils import mat4_perspective, mat4_rotation, mat4_translate
from spimagine_amd.volumerender.volumerender import render_matrices

pytestmark = pytest.mark.gpu

TOP = {np.uint16: 3000., np.uint8: 200., np.float32: 1.}


def volume(torch, kind, dtype, shape):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(3)

    def uniform(*s):
        return torch.rand(s, generator=gen, device="cuda")

    def normal(*s):
        return torch.randn(s, generator=gen, device="cuda")

    if kind == "noise":
        v = uniform(*shape)
    elif kind == "points":  # one voxel in 2,000 over nothing
        v = (uniform(*shape) > .9995) * uniform(*shape)
    elif kind == "grain":  # coarse noise over fine
        small = normal(1, 1, *[max(2, n // 8) for n in shape])
        v = torch.nn.functional.interpolate(small, size=shape, mode="trilinear")[0, 0]
        v = .5 + .15 * v + .02 * normal(*shape)
    elif kind == "noisy spots":
        v = torch.zeros(shape, device="cuda")
        rng = np.random.default_rng(4)
        for c in rng.integers(8, [n - 8 for n in shape], (int(np.prod(shape) / 50000.), 3)):
            z, y, x = [int(n) for n in c]
            v[z - 4:z + 5, y - 4:y + 5, x - 4:x + 5] += float(rng.uniform(.2, 1.))
        v = v + .1 + .3 * normal(*shape)
    v = (v * TOP[dtype]).clamp(0, 255 if dtype == np.uint8 else 32767)
    kinds = {np.uint16: torch.int16, np.uint8: torch.uint8, np.float32: torch.float32}
    return (v if dtype == np.float32 else v.round()).to(kinds[dtype]).contiguous()


def times(torch, s, ctx, go, chunks, key="chunk"):
    """The least time of each setting of a tuning key, taken in turn."""
    best = {k: 1e9 for k in chunks}
    for _ in range(7):
        for k in chunks:
            ctx.set_tuning(key, k)
            go()
            e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            e[0].record(s)
            for _ in range(4):
                go()
            e[1].record(s)
            e[1].synchronize()
            best[k] = min(best[k], e[0].elapsed_time(e[1]) * 250.)
    return best


# (how, voxel type, volume, shape, frame size, steps, frames)
ROUTES = [
    # bounds of empty float windows were widened above the ray's zero, and each was sampled
    ("frame", np.float32, "points", (256, 256, 256), 800, 448, 1),
    # more windows to sample than their gain paid for
    ("batch nearest", np.uint16, "noise", (256, 256, 256), 800, 200, 6),
    ("batch nearest", np.float32, "points", (128, 128, 128), 800, 200, 6),
    ("batch nearest", np.uint8, "grain", (192, 192, 192), 800, 200, 6),
    ("batch", np.uint16, "noisy spots", (256, 512, 512), 800, 200, 6),
    ("frame", np.uint16, "noisy spots", (384, 384, 384), 520, 200, 1),
    ("split", np.uint16, "noisy spots", (256, 512, 512), 200, 200, 6),
    ("split", np.uint8, "grain", (128, 128, 128), 200, 224, 6),
    # rays that cross the iso value at once, with look-ahead for many groups
    ("iso", np.uint8, "noise", (128, 128, 128), 1200, 112, 1),
    ("iso", np.float32, "noise", (128, 128, 128), 800, 200, 1),
]


@pytest.mark.parametrize("how,dtype,kind,shape,size,steps,n", ROUTES)
def test_default_march_is_not_slower(how, dtype, kind, shape, size, steps, n):
    import torch
    ctx = _lib.Context(0)
    vol = volume(torch, kind, dtype, shape)
    torch.cuda.synchronize()
    slot = ctx.volume_add(dev_ptr=vol.data_ptr(), dtype=dtype, shape=shape)
    s = torch.cuda.Stream()
    o = torch.zeros((n, 7, size, size), device="cuda")
    ps = []
    for k in range(n):
        M = np.dot(mat4_translate(0, 0, -3.2), mat4_rotation(.6 + .5 * k, .3, 1, -.2))
        iP, iM = render_matrices(M, mat4_perspective(45, 1., .1, 10), shape[::-1])
        ps.append(_lib.make_params(iP, iM, min_val=0., max_val=TOP[dtype], max_steps=steps,
                                   filter=_lib.FILTER_NEAREST if how.endswith("nearest") else
                                   _lib.FILTER_LINEAR))
    at = [[o[k, j].data_ptr() for j in range(5)] for k in range(n)]
    jobs = ctx.make_jobs([(slot, list(p.inv_p), list(p.inv_m), a[0], a[1]) for p, a in zip(ps, at)])
    frames = [_lib.make_frame(slot, p, size, size, a[0], a[1]) for p, a in zip(ps, at)]

    def go():
        st = s.cuda_stream
        if how.startswith("frame"):
            ctx.render_slot(slot, ps[0], _lib.METHOD_MAX_PROJECT, size, size, at[0][0], at[0][1], stream=st)
        elif how == "iso":
            ctx.render_slot(slot, ps[0], _lib.METHOD_ISO_SURFACE, size, size, at[0][0], at[0][1], at[0][2],
                            at[0][4], at[0][3], stream=st)
        elif how.startswith("batch"):
            ctx.render_batch(jobs, size, size, params=ps[0], stream=st)
        else:
            ctx.render_frames_split(frames, stream=st)

    torch.cuda.synchronize()
    outs = []
    for chunk in (0, 16):
        ctx.set_tuning("chunk", chunk)
        o.fill_(-1.)
        torch.cuda.synchronize()
        go()
        s.synchronize()
        outs.append(o.clone())
    assert torch.equal(outs[0], outs[1])
    best = times(torch, s, ctx, go, (0, 8, 16, 32))
    staged = min(v for k, v in best.items() if k)
    print("%s %s %s %s %d^2 %d steps: default %.0f us, staged %.0f us" % (
        how, np.dtype(dtype).name, kind, shape, size, steps, best[0], staged), flush=True)
    ctx.close()
    assert best[0] <= 1.2 * staged


# (voxel type, volume, shape, frame size, steps, frames, alpha_pow, bound of the time against no test)
OPACITY = [
    # windows asked where they could not end a ray: too few waves, a batch's still transparent rays
    (np.uint16, "noisy spots", (256, 256, 256), 400, 448, 1, .6, 1.07),
    (np.uint16, "noisy spots", (256, 256, 256), 400, 200, 1, .6, 1.07),
    (np.uint8, "noisy spots", (256, 256, 256), 400, 448, 6, .6, 1.07),
    (np.uint16, "noisy spots", (192, 192, 192), 400, 200, 6, .2, 1.07),
    # not asked, and the volume's own bounds end rays though voxels lie below min_val
    (np.uint16, "noise", (160, 160, 160), 200, 200, 1, .6, 1.),
    (np.uint8, "noise", (160, 160, 160), 600, 112, 1, .7, 1.),
    # asked: rays turn opaque, and voxels lie too far below min_val for the volume's bounds
    (np.uint16, "noise", (256, 256, 256), 800, 448, 1, .7, 1.),
    (np.uint16, "grain", (176, 176, 176), 400, 320, 6, .6, 1.),
    (np.float32, "grain", (176, 176, 176), 400, 320, 6, .6, 1.),
]


@pytest.mark.parametrize("dtype,kind,shape,size,steps,n,alpha_pow,bound", OPACITY)
def test_opacity_rays_end_early_where_that_pays(dtype, kind, shape, size, steps, n, alpha_pow, bound):
    import torch
    ctx = _lib.Context(0)
    vol = volume(torch, kind, dtype, shape)
    torch.cuda.synchronize()
    slot = ctx.volume_add(dev_ptr=vol.data_ptr(), dtype=dtype, shape=shape)
    s = torch.cuda.Stream()
    o = torch.zeros((n, 2, size, size), device="cuda")
    jobs = []
    for k in range(n):
        M = np.dot(mat4_translate(0, 0, -3.2), mat4_rotation(.6 + .5 * k, .3, 1, -.2))
        iP, iM = render_matrices(M, mat4_perspective(45, 1., .1, 10), shape[::-1])
        p = _lib.make_params(iP, iM, min_val=.08 * TOP[dtype], max_val=.9 * TOP[dtype], max_steps=steps,
                             alpha_pow=alpha_pow)
        jobs.append((slot, list(p.inv_p), list(p.inv_m), o[k, 0].data_ptr(), o[k, 1].data_ptr()))
    frame = (slot, p, _lib.METHOD_MAX_PROJECT, size, size, o[0, 0].data_ptr(), o[0, 1].data_ptr())
    jobs = ctx.make_jobs(jobs)

    def go():
        if n == 1:
            ctx.render_slot(*frame, stream=s.cuda_stream)
        else:
            ctx.render_batch(jobs, size, size, params=p, stream=s.cuda_stream)

    outs = []
    for skip in (0, 1):
        ctx.set_tuning("skip", skip)
        o.fill_(-1.)
        torch.cuda.synchronize()
        go()
        s.synchronize()
        outs.append(o.clone())
    assert torch.equal(outs[0], outs[1])
    best = times(torch, s, ctx, go, (0, 1), "skip")
    print("opacity %s %s %s %d^2 %d steps, %d: %.0f us, without the test %.0f us" % (
        np.dtype(dtype).name, kind, shape, size, steps, n, best[1], best[0]), flush=True)
    ctx.close()
    assert best[1] <= bound * best[0]
