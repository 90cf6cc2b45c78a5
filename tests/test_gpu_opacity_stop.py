"""GPU: the opacity mode that stops once the window grid shows that no later sample can raise
a ray's colour, against the same frames with every box sampled (SPR_TUNE_SKIP 0), bit for bit."""
import numpy as np
import pytest

from spimagine_amd import _lib, synth
from spimagine_amd.utils import mat4_perspective, mat4_rotation, mat4_translate
from spimagine_amd.volumerender.volumerender import render_matrices

pytestmark = pytest.mark.gpu

POSES = [np.dot(mat4_translate(0, 0, -3.4), mat4_rotation(.7, .3, 1, -.2)),
         np.dot(mat4_translate(.2, -.1, -2.2), mat4_rotation(2.3, 1, .2, .5))]  # enters the volume
BOXES = [(-1, 1, -1, 1, -1, 1), (-1.6, 1.7, -1.2, 1, -1, 2.)]
SCALE = {np.uint8: 200., np.uint16: 3000., np.float32: 1.}


def volume(dtype, shape, seed):
    top = SCALE[dtype]
    vol = synth.blob_volume(shape, n_blobs=14, sigma=(2., 6.), amp=(.3 * top, top),
                            background=.08 * top, poisson=False, read_noise=.02 * top, dtype=dtype,
                            seed=seed)
    if dtype == np.float32:
        vol[shape[0] // 2, shape[1] // 3] = np.nan
        vol[shape[0] // 4, 2, 3] = np.inf
        vol[shape[0] // 4, 9, 3] = -np.inf
    return vol


# (min, max) of the transfer as shares of the brightest voxel: noise reaches below min_val,
# everything above it, a falling range, no normalisation, a range so narrow that a step's
# factor turns negative
RANGES = [(.1, .7), (0., 1.), (.8, .1), (.1, 0.), (.3, .3004)]


# frames large enough to ask the windows: boxes of 16, 8 and 4 samples, a march of one sample an
# epoch and one of many; a volume too small to
@pytest.mark.parametrize("dtype", [np.uint16, np.uint8, np.float32])
@pytest.mark.parametrize("shape,steps", [((64, 64, 256), 224), ((60, 170, 50), 112),
                                         ((33, 90, 160), 18), ((30, 31, 161), 1700),
                                         ((40, 41, 50), 96)])
@pytest.mark.parametrize("filt", [0, 1])
def test_stopped_rays_keep_their_colour(dtype, shape, steps, filt):
    import torch
    ctx = _lib.Context(0)
    W, H = 401, 343
    top = SCALE[dtype]
    slot = ctx.volume_add(volume(dtype, shape, 4))
    P = mat4_perspective(45, W / float(H), .1, 10)
    s = torch.cuda.Stream()
    for k, (M, box) in enumerate(zip(POSES, BOXES)):
        iP, iM = render_matrices(M, P, shape[::-1], (1., 1., 1.4))
        for lo, hi in RANGES:
            for ap in (.2, 1., 3.):
                p = _lib.make_params(iP, iM, box, np.float32(lo * top), np.float32(hi * top),
                                     alpha_pow=ap, max_steps=steps, filter=filt)
                outs = []
                for skip in (1, 0):
                    ctx.set_tuning("skip", skip)
                    o = torch.full((2, H, W), -7., device="cuda")
                    torch.cuda.synchronize()  # (filled before the other stream writes)
                    ctx.render_slot(slot, p, _lib.METHOD_MAX_PROJECT, W, H, o[0].data_ptr(),
                                    o[1].data_ptr(), stream=s.cuda_stream)
                    s.synchronize()
                    outs.append(o.cpu().numpy())
                what = "pose %d range %g %g alpha_pow %g" % (k, lo, hi, ap)
                np.testing.assert_array_equal(outs[0], outs[1], err_msg=what)
                ctx.set_tuning("skip", 1)
                b = torch.full((2, H, W), -7., device="cuda")
                torch.cuda.synchronize()
                ctx.render_batch([(slot, list(iP), list(iM), b[0].data_ptr(), b[1].data_ptr())], W, H,
                                 params=p, stream=s.cuda_stream)
                s.synchronize()
                np.testing.assert_array_equal(b.cpu().numpy(), outs[1], err_msg="batch, " + what)
