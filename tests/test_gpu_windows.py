"""GPU: the max projection gathered group by group by the window grid (the default where it
pays) against the same frame with every sample taken from global memory (SPR_TUNE_SLAB_KB 0)
and against the oracle, bit for bit."""
import numpy as np
import pytest

import oracle
from spimagine_amd import _lib, synth
from spimagine_amd.utils import mat4_perspective, mat4_rotation, mat4_translate
from spimagine_amd.volumerender.volumerender import render_matrices

pytestmark = pytest.mark.gpu

POSES = [np.dot(mat4_translate(0, 0, -3.4), mat4_rotation(.7, .3, 1, -.2)),
         np.dot(mat4_translate(.2, -.1, -2.2), mat4_rotation(2.3, 1, .2, .5)),  # enters the volume
         np.dot(mat4_translate(0, 0, -4.), mat4_rotation(0., 0, 1, 0))]  # along the axes
BOXES = [(-1, 1, -1, 1, -1, 1), (-.7, .4, -1, .9, -.2, 1), (-1.6, 1.7, -1.2, 1, -1, 2.)]


def volume(dtype, shape, seed):
    amp, bg = {np.uint8: ((60., 200.), 6.), np.uint16: ((500., 3000.), 100.),
               np.float32: ((.3, 1.), -.1)}[dtype]
    return synth.blob_volume(shape, n_blobs=14, sigma=(2., 5.), amp=amp, background=bg,
                             poisson=False, read_noise=.02 * amp[1], dtype=dtype, seed=seed)


def render(torch, ctx, slot, p, W, H):
    o = torch.full((2, H, W), -7., device="cuda")
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    ctx.render_slot(slot, p, _lib.METHOD_MAX_PROJECT, W, H, o[0].data_ptr(), o[1].data_ptr(),
                    stream=s.cuda_stream)
    s.synchronize()
    return o.cpu().numpy()


# steps: 4, 2 and 1 samples a group (0.6, 1.3 and 5 voxels a step), one box, segments without
# samples (16 steps), long rays
@pytest.mark.parametrize("dtype", [np.uint16, np.uint8, np.float32])
@pytest.mark.parametrize("shape,steps", [((64, 64, 128), 224), ((60, 117, 50), 112),
                                         ((64, 128, 32), 96), ((33, 90, 130), 18),
                                         ((50, 40, 112), 16), ((30, 31, 113), 1700)])
def test_windows_equal_every_sample(dtype, shape, steps):
    import torch
    ctx = _lib.Context(0)
    W, H = 117, 75
    vol = volume(dtype, shape, 5)
    if dtype == np.float32:
        vol[shape[0] // 2, shape[1] // 3] = np.nan
        vol[shape[0] // 4, 2, 3] = np.inf
    slot = ctx.volume_add(vol)
    P = mat4_perspective(45, W / float(H), .1, 10)
    for k, (M, box) in enumerate(zip(POSES, BOXES)):
        iP, iM = render_matrices(M, P, shape[::-1], (1., 1., 1.5))
        p = _lib.make_params(iP, iM, box, .02, 900. if dtype == np.uint16 else 150. if
                             dtype == np.uint8 else .9, gamma=(1., .6, 1.)[k], max_steps=steps)
        ctx.set_tuning("slab_kb", 19)
        got = render(torch, ctx, slot, p, W, H)
        ctx.set_tuning("slab_kb", 0)
        np.testing.assert_array_equal(got, render(torch, ctx, slot, p, W, H), err_msg=str(k))
        assert (got[1] > 0).sum() > 100


def test_windows_against_the_oracle():
    import torch
    ctx = _lib.Context(0)
    vol = volume(np.uint16, (80, 70, 116), 8)
    W, H = 90, 66
    iP, iM = render_matrices(POSES[0], mat4_perspective(45, W / float(H), .1, 10), (116, 70, 80))
    p = _lib.make_params(iP, iM, (-1, 1, -1, 1, -1, 1), 100., 2500., max_steps=160)
    got = render(torch, ctx, ctx.volume_add(vol), p, W, H)
    out, alpha = oracle.max_project(vol, iP, iM, min_val=100., max_val=2500., max_steps=160,
                                    width=W, height=H)
    np.testing.assert_array_equal(got[0], out)
    np.testing.assert_array_equal(got[1], alpha)


def test_noise_is_staged():
    """White noise leaves nothing to skip: the frame stays with the staged kernel, and equals
    the gathered one's samples."""
    import torch
    rng = np.random.default_rng(3)
    ctx = _lib.Context(0)
    vol = rng.integers(0, 4000, (64, 60, 120)).astype(np.uint16)
    W, H = 100, 90
    iP, iM = render_matrices(POSES[1], mat4_perspective(45, W / float(H), .1, 10), (120, 60, 64))
    for steps in (112, 24):
        p = _lib.make_params(iP, iM, (-1, 1, -1, 1, -1, 1), 0., 4000., max_steps=steps)
        slot = ctx.volume_add(vol)
        ctx.set_tuning("slab_kb", 19)
        got = render(torch, ctx, slot, p, W, H)
        ctx.set_tuning("slab_kb", 0)
        np.testing.assert_array_equal(got, render(torch, ctx, slot, p, W, H))


def test_batches_gathered_and_staged():
    """A uniform batch and a mixed one by the window grid (the default for small frames),
    from the persistent queues (SPR_TUNE_CHUNK 16), without allocation and as a graph: the
    frames of each rendered alone, bit for bit."""
    import torch
    ctx = _lib.Context(0)
    vols = [volume(np.uint16, s, k) for k, s in enumerate(((40, 50, 112), (33, 64, 41), (70, 30, 52)))]
    slots = [ctx.volume_add(v) for v in vols]
    W, H = 75, 93
    sizes, ps, want = [], [], []
    for k in range(7):
        v = k % 3
        w, h = (W, H) if k < 4 else (16 * k, 131 - 17 * k)
        iP, iM = render_matrices(POSES[k % 3], mat4_perspective(45, w / float(h), .1, 10),
                                 vols[v].shape[::-1])
        p = _lib.make_params(iP, iM, BOXES[0 if k < 4 else k % 3], 50., 2000.,
                             max_steps=96 if k < 4 else (16, 40, 200)[k % 3])
        sizes.append((v, w, h))
        ps.append(p)
        want.append(render(torch, ctx, slots[v], p, w, h))
    s = torch.cuda.Stream()

    def check(launch, ks):
        outs = [torch.full((2, sizes[k][2], sizes[k][1]), -9., device="cuda") for k in ks]
        launch(outs, ks)
        s.synchronize()
        for o, k in zip(outs, ks):
            np.testing.assert_array_equal(o.cpu().numpy(), want[k], err_msg=str(k))

    def jobs(outs, ks):
        return [(slots[sizes[k][0]], list(ps[k].inv_p), list(ps[k].inv_m), o[0].data_ptr(),
                 o[1].data_ptr()) for o, k in zip(outs, ks)]

    def batch(outs, ks):
        ctx.render_batch(jobs(outs, ks), W, H, params=ps[0], stream=s.cuda_stream)

    def noalloc(outs, ks):
        ctx.render_batch_noalloc(jobs(outs, ks), W, H, params=ps[0], stream=s.cuda_stream)

    def frames(outs, ks):
        ctx.render_frames([_lib.make_frame(slots[sizes[k][0]], ps[k], sizes[k][1], sizes[k][2],
                                           o[0].data_ptr(), o[1].data_ptr())
                           for o, k in zip(outs, ks)], stream=s.cuda_stream)

    def graph(outs, ks):
        p = ps[0]
        ctx.lib.spr_set_params(ctx.handle, p)
        g = ctx.batch_graph(jobs(outs, ks), W, H)
        for o in outs:  # replayed after other work on the outputs
            g.launch(s.cuda_stream)
            s.synchronize()
            o.fill_(3.)
            torch.cuda.synchronize()
        g.launch(s.cuda_stream)
        s.synchronize()
        g.close()

    for chunk in (0, 16):
        ctx.set_tuning("chunk", chunk)
        for f in (batch, noalloc, graph):
            check(f, range(4))
        check(frames, range(7))
        check(frames, [6])


@pytest.mark.parametrize("dtype,filt", [(np.uint16, 0), (np.uint8, 0), (np.float32, 0),
                                        (np.uint16, 1), (np.float32, 1)])
@pytest.mark.parametrize("shape,steps", [((64, 64, 64), 150), ((60, 77, 50), 75), ((33, 90, 70), 17),
                                         ((40, 41, 50), 2), ((30, 31, 29), 2100)])
def test_iso_windows_equal_every_sample(dtype, filt, shape, steps):
    """The iso surface by the window grid against the march with every sample from global
    memory: all five outputs, from outside and inside the volume, iso values that the first
    sample lies above and below, a NaN row, one and many runs of groups (4, 2 and 1 samples a
    group; the least number of steps; more than one anchor along a ray)."""
    import torch
    ctx = _lib.Context(0)
    W, H = 101, 83
    vol = volume(dtype, shape, 6)
    if dtype == np.float32:
        vol[shape[0] // 2, shape[1] // 3] = np.nan
    slot = ctx.volume_add(vol)
    P = mat4_perspective(45, W / float(H), .1, 10)
    top = float(np.nanmax(vol))
    for k, (M, box) in enumerate(zip(POSES, BOXES)):
        iP, iM = render_matrices(M, P, shape[::-1], (1., 1., 1.3))
        for level in (.25, .02 if k else 1.6):
            p = _lib.make_params(iP, iM, box, 0., top * level * 2, max_steps=steps, occ_radius=5,
                                 filter=filt)
            outs = {}
            for slab in (19, 0):
                ctx.set_tuning("slab_kb", slab)
                o = [torch.full((H, W), -7., device="cuda") for _ in range(4)]
                n = torch.full((H, W, 3), -7., device="cuda")
                s = torch.cuda.Stream()
                ctx.render_slot(slot, p, _lib.METHOD_ISO_SURFACE, W, H, o[0].data_ptr(),
                                o[1].data_ptr(), o[2].data_ptr(), n.data_ptr(), o[3].data_ptr(),
                                stream=s.cuda_stream)
                s.synchronize()
                outs[slab] = [t.cpu().numpy() for t in o + [n]]
            for a, b in zip(outs[19], outs[0]):
                np.testing.assert_array_equal(a, b, err_msg="pose %d level %g" % (k, level))


@pytest.mark.parametrize("dtype", [np.uint16, np.uint8, np.float32])
@pytest.mark.parametrize("shape,steps", [((64, 64, 128), 224), ((60, 117, 50), 112),
                                         ((33, 90, 130), 18), ((30, 31, 113), 1700)])
def test_nearest_windows_equal_every_sample(dtype, shape, steps):
    """The nearest filter by the window grid (4, 2 and 1 samples a group, long rays; a frame
    alone, a uniform and a mixed batch) against every sample from global memory."""
    import torch
    ctx = _lib.Context(0)
    W, H = 117, 75
    vol = volume(dtype, shape, 7)
    if dtype == np.float32:
        vol[shape[0] // 2, shape[1] // 3] = np.nan
        vol[shape[0] // 4, 2, 3] = np.inf
    slot = ctx.volume_add(vol)
    P = mat4_perspective(45, W / float(H), .1, 10)
    for k, (M, box) in enumerate(zip(POSES, BOXES)):
        iP, iM = render_matrices(M, P, shape[::-1], (1., 1., 1.5))
        p = _lib.make_params(iP, iM, box, .02, 900. if dtype == np.uint16 else 150. if
                             dtype == np.uint8 else .9, gamma=(1., .6, 1.)[k], max_steps=steps,
                             filter=_lib.FILTER_NEAREST)
        s = torch.cuda.Stream()
        outs = []
        for slab in (19, 0):
            ctx.set_tuning("slab_kb", slab)
            o = torch.full((3, 2, H, W), -7., device="cuda")
            torch.cuda.synchronize()
            ctx.render_slot(slot, p, _lib.METHOD_MAX_PROJECT, W, H, o[0, 0].data_ptr(),
                            o[0, 1].data_ptr(), stream=s.cuda_stream)
            ctx.render_batch([(slot, list(iP), list(iM), o[1, 0].data_ptr(), o[1, 1].data_ptr())],
                             W, H, params=p, stream=s.cuda_stream)
            ctx.render_frames([_lib.make_frame(slot, p, W, H, o[2, 0].data_ptr(), o[2, 1].data_ptr())],
                              stream=s.cuda_stream, filter=_lib.FILTER_NEAREST)
            s.synchronize()
            outs.append(o.cpu().numpy())
        np.testing.assert_array_equal(outs[0], outs[1], err_msg=str(k))
        assert (outs[0][:, 1] > 0).sum() > 300
        np.testing.assert_array_equal(outs[0][0], outs[0][1])
        np.testing.assert_array_equal(outs[0][0], outs[0][2])


# the pooled volume's rays take 4, 2 and 1 samples a group, in one box or two passes
@pytest.mark.parametrize("shape,steps,parts", [((128, 64, 256), 224, 1), ((60, 117, 230), 96, 1),
                                               ((66, 41, 231), 18, 1), ((61, 50, 241), 640, 2)])
def test_pair_windows_equal_staged(shape, steps, parts):
    """Both channels of a pooled pair by the window grid against the staged boxes
    (SPR_TUNE_CHUNK 16): from outside and inside the volume, boxes past it."""
    import torch
    ctx = _lib.Context(0)
    pair = ctx.volume_add_pooled_pair(ctx.volume_add(volume(np.uint16, shape, 9)))
    nz, ny, nx = ctx.volume_info(pair)["shape"]
    W, H = 119, 86
    P = mat4_perspective(45, W / float(H), .1, 10)
    s = torch.cuda.Stream()
    for k, (M, box) in enumerate(zip(POSES, BOXES)):
        iP, iM = render_matrices(M, P, (nx, ny, nz), (1., 1., 1.5))
        p = _lib.make_params(iP, iM, box, 100., 2500., max_steps=steps)
        outs = []
        for chunk in (0, 16):
            ctx.set_tuning("chunk", chunk)
            o = torch.full((3, H, W), -7., device="cuda")
            torch.cuda.synchronize()
            for part in range(parts):
                ctx.render_pair(pair, p, W, H, o[0].data_ptr(), o[2].data_ptr(), num_parts=parts,
                                current_part=part, stream=s.cuda_stream)
            s.synchronize()
            outs.append(o.cpu().numpy())
        np.testing.assert_array_equal(outs[0], outs[1], err_msg=str(k))
        assert (outs[0][1] > 0).sum() > 300
