"""GPU: the upload path (padded copy, window grid and brick bounds in one pass, host volumes a
slab of planes at a time): the resident voxels, the volume's bounds and the frames of a host
upload, a device upload and a linear-layout slot agree."""
import numpy as np
import pytest

from spimagine_amd import _lib
from spimagine_amd.utils import mat4_perspective, mat4_rotation, mat4_translate
from spimagine_amd.volumerender.volumerender import render_matrices

pytestmark = pytest.mark.gpu

# one voxel, rows shorter than a 16-byte unit, one past and one short of 4-voxel blocks and
# 16-byte units, many units a row; the last one is larger than one slab of the staged upload
SHAPES = [(1, 1, 1), (2, 3, 5), (7, 6, 14), (9, 13, 33), (30, 31, 62), (5, 70, 257)]
BIG = (210, 401, 420)


def frames(torch, ctx, slot, shape, lo, hi, W=90, H=70):
    P = mat4_perspective(45, W / float(H), .1, 10)
    M = np.dot(mat4_translate(0, 0, -3.2), mat4_rotation(.8, .4, 1, .3))
    iP, iM = render_matrices(M, P, shape[::-1])
    p = _lib.make_params(iP, iM, (-1, 1, -1, 1, -1, 1), lo, hi, max_steps=160)
    o = torch.full((2, H, W), -3., device="cuda")
    s = torch.cuda.Stream()
    ctx.render_slot(slot, p, _lib.METHOD_MAX_PROJECT, W, H, o[0].data_ptr(), o[1].data_ptr(),
                    stream=s.cuda_stream)
    s.synchronize()
    return o.cpu().numpy()


def check(torch, vol):
    ctx = _lib.Context(0)
    lo, hi = float(vol.min()), float(vol.max()) + 1.
    ctx.set_layout(_lib.LAYOUT_LINEAR)
    ref = ctx.volume_add(vol)
    want = frames(torch, ctx, ref, vol.shape, lo, hi)
    ctx.set_layout(_lib.LAYOUT_PADDED)
    dev = torch.from_numpy(vol.view(np.int16) if vol.dtype == np.uint16 else vol).cuda()
    slots = [ctx.volume_add(vol), ctx.volume_add(dev_ptr=dev.data_ptr(), dtype=vol.dtype,
                                                 shape=vol.shape)]
    for slot in slots:
        np.testing.assert_array_equal(ctx.volume_read(slot), vol)
        np.testing.assert_array_equal(frames(torch, ctx, slot, vol.shape, lo, hi), want)
    ctx.set_volume(vol)
    ctx.set_volume(vol[::-1].copy())  # refilled in place
    np.testing.assert_array_equal(ctx.volume_read(0), vol[::-1])
    assert ctx.volume_minmax() == (float(vol.min()), float(vol.max()))
    assert (want[1] > 0).any()


@pytest.mark.parametrize("dtype", [np.uint16, np.uint8, np.float32])
@pytest.mark.parametrize("shape", SHAPES)
def test_upload_small_and_ragged(dtype, shape):
    import torch
    rng = np.random.default_rng(sum(shape))
    top = 255 if dtype == np.uint8 else 40000
    check(torch, (rng.uniform(0, 1, shape) ** 6 * top).astype(dtype))


@pytest.mark.parametrize("dtype", [np.uint16, np.float32])
def test_upload_in_several_slabs(dtype):
    import torch
    rng = np.random.default_rng(7)
    vol = (rng.random(BIG, np.float32) ** 8 * 3000.).astype(dtype)
    assert vol.nbytes > 64 << 20
    check(torch, vol)
