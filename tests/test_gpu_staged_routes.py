"""GPU: the staged kernels that the default tuning leaves for volumes with little to skip -- and
that a chunk length (SPR_TUNE_CHUNK) asks for on any volume -- against the same frames with every
sample taken from global memory, bit for bit: segments of scattered rays, the one-wave march of
volumes above 4 GiB, the one-wave iso march that skips bricks, and the opacity mode that asks the
windows of such a volume."""
import numpy as np
import pytest

from spimagine_amd import _lib, learned, synth
from spimagine_amd.utils import mat4_perspective, mat4_rotation, mat4_translate
from spimagine_amd.volumerender.volumerender import render_matrices

pytestmark = pytest.mark.gpu

POSES = [np.dot(mat4_translate(0, 0, -3.2), mat4_rotation(.7, .3, 1, -.2)),
         np.dot(mat4_translate(.5, -.3, -2.6), mat4_rotation(2.3, 1, .2, .5)),  # rays miss
         np.dot(mat4_translate(0, 0, -4.), mat4_rotation(0., 0, 1, 0))]
TOP = {np.uint16: 3000., np.uint8: 200., np.float32: 1.}


def blobs(dtype, shape, seed):
    top = TOP[dtype]
    return synth.blob_volume(shape, n_blobs=12, sigma=(2., 5.), amp=(.2 * top, top),
                             background=.04 * top, poisson=False, read_noise=.02 * top, dtype=dtype,
                             seed=seed)


def noise(dtype, shape, seed):
    v = np.random.default_rng(seed).uniform(.1, 1., shape) * TOP[dtype]
    return v.astype(dtype)


# chunk 16: staged whatever the volume holds; noise: staged by default
@pytest.mark.parametrize("dtype", [np.uint16, np.uint8, np.float32])
@pytest.mark.parametrize("seg", [32, 64, 128])
@pytest.mark.parametrize("make,chunk", [(blobs, 16), (noise, 0)])
def test_staged_segments_of_scattered_rays(dtype, seg, make, chunk):
    import torch
    ctx = _lib.Context(0)
    vol = make(dtype, (44, 61, 53), seg)
    slot = ctx.volume_add(vol)
    lo, hi = float(vol.min()), float(vol.max())
    s = torch.cuda.Stream()
    frames = []
    for w, h, k, steps, span, box, stride in [
            (128, 96, 0, 160, (lo, hi, 1.), (-1, 1, -1, 1, -1, 1), 8),
            (256, 128, 1, 96, (0., 0., 1.), (-1, 1, -1, 1, -1, 1), 16),
            (77, 45, 2, 208, (lo, hi, .7), (-1, 1, -.6, .8, -1, .5), 0)]:
        iP, iM = render_matrices(POSES[k], mat4_perspective(45, w / float(h), .1, 10), vol.shape[::-1])
        p = _lib.make_params(iP, iM, box, *span, max_steps=steps)
        if stride:
            p = learned.sparse_params(p, w, h, stride=stride)
            w, h = w // stride, h // stride
        frames.append((p, w, h, torch.full((4, h, w), -7., device="cuda")))
    torch.cuda.synchronize()
    ctx.set_tuning("slab_kb", 0)
    for p, w, h, o in frames:
        ctx.render_slot(slot, p, _lib.METHOD_MAX_PROJECT, w, h, o[0].data_ptr(), o[1].data_ptr(),
                        stream=s.cuda_stream)
    ctx.set_tuning("slab_kb", 19)
    ctx.set_tuning("chunk", chunk)
    ctx.render_frames_split([_lib.make_frame(slot, p, w, h, o[2].data_ptr(), o[3].data_ptr())
                             for p, w, h, o in frames], seg=seg, stream=s.cuda_stream)
    s.synchronize()
    for k, (p, w, h, o) in enumerate(frames):
        o = o.cpu().numpy()
        np.testing.assert_array_equal(o[2:], o[:2], err_msg="frame %d" % k)
        assert (o[0] > 0).sum() > 20
    ctx.close()


def iso(torch, ctx, slot, p, W, H, s):
    o = [torch.full((H, W), -7., device="cuda") for _ in range(4)]
    n = torch.full((H, W, 3), -7., device="cuda")
    torch.cuda.synchronize()
    ctx.render_slot(slot, p, _lib.METHOD_ISO_SURFACE, W, H, o[0].data_ptr(), o[1].data_ptr(),
                    o[2].data_ptr(), n.data_ptr(), o[3].data_ptr(), stream=s.cuda_stream)
    s.synchronize()
    return o + [n]


@pytest.mark.parametrize("dtype", [np.uint16, np.uint8, np.float32])
@pytest.mark.parametrize("shape,steps", [((64, 64, 64), 150), ((60, 77, 50), 75), ((33, 90, 70), 17)])
def test_staged_iso_march_skips_bricks(dtype, shape, steps):
    import torch
    ctx = _lib.Context(0)
    W, H = 101, 83
    vol = blobs(dtype, shape, 6)
    if dtype == np.float32:
        vol[shape[0] // 2, shape[1] // 3] = np.nan
    slot = ctx.volume_add(vol)
    s = torch.cuda.Stream()
    top = float(np.nanmax(vol))
    hits = 0
    for k, M in enumerate(POSES):
        iP, iM = render_matrices(M, mat4_perspective(45, W / float(H), .1, 10), shape[::-1])
        for level in (.25, .04):
            p = _lib.make_params(iP, iM, max_val=2. * level * top, max_steps=steps, occ_radius=5)
            ctx.set_tuning("chunk", 0)
            ctx.set_tuning("slab_kb", 0)
            want = iso(torch, ctx, slot, p, W, H, s)
            ctx.set_tuning("slab_kb", 19)
            hits += int(torch.isfinite(want[2]).sum())
            for chunk in (16, 8, 4):
                ctx.set_tuning("chunk", chunk)
                for a, b in zip(iso(torch, ctx, slot, p, W, H, s), want):
                    np.testing.assert_array_equal(a.cpu().numpy(), b.cpu().numpy(),
                                                  err_msg="pose %d level %g chunk %d" % (k, level, chunk))
    assert hits > 500
    ctx.close()


def test_volume_above_4_gib_staged_and_by_windows():
    import torch
    shape = (512, 2048, 2048)
    v16 = next(synth.blob_series_device(shape, 3000, (3., 10.), (500., 3000.), 100., False, 5., 1, seed=3))
    torch.cuda.synchronize()
    wide, lin = _lib.Context(0), _lib.Context(0)
    lin.set_layout(_lib.LAYOUT_LINEAR)
    sw, sl = [c.volume_add(dev_ptr=v16.data_ptr(), dtype=np.uint16, shape=shape) for c in (wide, lin)]
    del v16
    s = torch.cuda.Stream()
    W, H = 528, 512  # 4,224 quarters: opacity frames ask the windows

    def mip(ctx, slot, p):
        o = torch.full((2, H, W), -7., device="cuda")
        torch.cuda.synchronize()
        ctx.render_slot(slot, p, _lib.METHOD_MAX_PROJECT, W, H, o[0].data_ptr(), o[1].data_ptr(),
                        stream=s.cuda_stream)
        s.synchronize()
        return o

    for k, M in enumerate(POSES[:2]):
        iP, iM = render_matrices(M, mat4_perspective(45, W / float(H), .1, 10), shape[::-1])
        for steps, ap in ((208, 0.), (2688, 0.), (2688, .6), (1360, 2.)):
            p = _lib.make_params(iP, iM, min_val=90., max_val=3300., alpha_pow=ap, max_steps=steps)
            want = mip(lin, sl, p)
            assert (want[0] > 0).sum().item() > 5000
            for chunk in (0, 16) if ap else (0, 4, 8, 16, 32):
                wide.set_tuning("chunk", chunk)
                assert torch.equal(mip(wide, sw, p), want), (k, steps, ap, chunk)
        p = _lib.make_params(iP, iM, max_val=3000., max_steps=2016)
        want = iso(torch, lin, sl, p, W, H, s)
        for chunk in (0, 16):
            wide.set_tuning("chunk", chunk)
            for a, b in zip(iso(torch, wide, sw, p, W, H, s), want):
                assert torch.equal(a, b), (k, chunk)
    wide.close()
    lin.close()
