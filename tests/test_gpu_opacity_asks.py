"""GPU: single opacity frames of enough waves to ask the window grid what is still to come (batches
of smaller ones do that in test_gpu_opacity_stop.py), against every box sampled, bit for bit."""
import numpy as np
import pytest

from spimagine_amd import _lib
from spimagine_amd.utils import mat4_perspective
from spimagine_amd.volumerender.volumerender import render_matrices
from test_gpu_opacity_stop import BOXES, POSES, RANGES, SCALE, volume

pytestmark = pytest.mark.gpu


# 5,412 quarters: boxes of 16, 8 and 4 samples, a march of one sample an epoch and one of many
@pytest.mark.parametrize("dtype", [np.uint16, np.uint8, np.float32])
@pytest.mark.parametrize("shape,steps", [((64, 64, 256), 224), ((60, 170, 50), 112),
                                         ((33, 90, 160), 80), ((30, 31, 161), 1700)])
@pytest.mark.parametrize("filt", [0, 1])
def test_asking_frames_keep_their_colours(dtype, shape, steps, filt):
    import torch
    ctx = _lib.Context(0)
    W, H = 641, 513
    top = SCALE[dtype]
    slot = ctx.volume_add(volume(dtype, shape, 4))
    s = torch.cuda.Stream()
    o = torch.empty((2, 2, H, W), device="cuda")
    for k, (M, box) in enumerate(zip(POSES, BOXES)):
        iP, iM = render_matrices(M, mat4_perspective(45, W / float(H), .1, 10), shape[::-1], (1., 1., 1.4))
        for lo, hi in RANGES:
            for ap in (.2, 1., 3.):
                p = _lib.make_params(iP, iM, box, np.float32(lo * top), np.float32(hi * top),
                                     alpha_pow=ap, max_steps=steps, filter=filt)
                o.fill_(-7.)
                torch.cuda.synchronize()  # (filled before the other stream writes)
                for skip in (1, 0):
                    ctx.set_tuning("skip", skip)
                    ctx.render_slot(slot, p, _lib.METHOD_MAX_PROJECT, W, H, o[skip, 0].data_ptr(),
                                    o[skip, 1].data_ptr(), stream=s.cuda_stream)
                s.synchronize()
                assert torch.equal(o[0].view(torch.int32), o[1].view(torch.int32)), (k, lo, hi, ap)
    ctx.close()


@pytest.mark.parametrize("dtype", [np.uint16, np.float32])
def test_small_frames_beside_one_that_asks(dtype):
    """Frames of their own sizes in one launch: all of them ask once one does, those of a few
    voxels, pixels and samples too."""
    import torch
    ctx = _lib.Context(0)
    rng = np.random.default_rng(5)
    top = SCALE[dtype]
    s = torch.cuda.Stream()
    specs = [((176, 170, 176), 480, 400, 320)] + [
        (shape, w, h, n) for shape, (w, h, n) in zip(
            [(1, 1, 1), (3, 4, 5), (2, 7, 8), (9, 3, 30), (33, 6, 14), (60, 61, 15)],
            [(33, 21, 16), (16, 16, 17), (64, 65, 40), (200, 7, 96), (90, 90, 300), (128, 100, 1100)])]
    frames, want = [], []
    for k, (shape, w, h, steps) in enumerate(specs):
        v = (top * rng.uniform(0, 1, shape)).astype(dtype)
        slot = ctx.volume_add(v)
        iP, iM = render_matrices(POSES[k % 2], mat4_perspective(45, w / float(h), .1, 10), shape[::-1])
        p = _lib.make_params(iP, iM, min_val=.08 * top, max_val=.9 * top, alpha_pow=.6, max_steps=steps)
        a, b = (torch.full((2, h, w), -7., device="cuda") for _ in range(2))
        torch.cuda.synchronize()
        ctx.set_tuning("skip", 0)
        ctx.render_slot(slot, p, _lib.METHOD_MAX_PROJECT, w, h, a[0].data_ptr(), a[1].data_ptr(),
                        stream=s.cuda_stream)
        frames.append((_lib.make_frame(slot, p, w, h, b[0].data_ptr(), b[1].data_ptr()), b))
        want.append(a)
    ctx.set_tuning("skip", 1)
    ctx.render_frames([f for f, _ in frames], alpha_pow=.6, stream=s.cuda_stream)
    s.synchronize()
    for (_, b), a, spec in zip(frames, want, specs):
        assert torch.equal(a, b), spec
    ctx.close()
