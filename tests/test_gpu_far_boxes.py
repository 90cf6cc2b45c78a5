"""GPU: the max projection by the window grid in boxes that reach far past the volume, where a
position estimated ahead of the running sum is off by the rounding of large positions, against
the same frame with every sample taken (SPR_TUNE_SLAB_KB 0), bit for bit."""
import numpy as np
import pytest

from spimagine_amd import _lib

pytestmark = pytest.mark.gpu

NX = 65000
# (box from -a to b along x, bright voxel): boxes whose rays take one sample between voxels v and
# v + 1 which the window estimated 8 to 15 samples before starts two voxels too late for (float32
# steps of 7.8 volumes from -a on, replayed on the host)
FAR = [(1575.1806640625, 1841.7265625, 25985), (1811.744140625, 1622.3193359375, 6085),
       (1580.9599609375, 1847.849609375, 16509), (1997.39453125, 1578.8759765625, 41929),
       (1794.3212890625, 1606.8525390625, 8741), (1871.6884765625, 1929.2666015625, 3141),
       (1904.2509765625, 1708.31640625, 58893), (1885.525390625, 1913.6796875, 7769)]


@pytest.mark.parametrize("filt", [0, 1])
@pytest.mark.parametrize("mixed", [False, True])
def test_samples_far_from_the_box_are_asked_for(filt, mixed):
    import torch
    W = H = 8
    inv_p = np.zeros((4, 4), np.float32)  # parallel rays along x
    inv_p[0, 2], inv_p[1, 0], inv_p[2, 1], inv_p[3, 3] = 4096., .5, .5, 1.
    for a, b, v in FAR:
        vol = np.zeros((4, 4, NX), np.uint16)
        vol[:, :, v:v + 2] = 3000
        ctx = _lib.Context(0)
        slot = ctx.volume_add(vol)
        p = _lib.make_params(inv_p, np.eye(4), (-a, b, -1, 1, -1, 1), max_val=6000., max_steps=256,
                             filter=filt)
        outs = []
        for slab in (19, 0):
            ctx.set_tuning("slab_kb", slab)
            o = torch.full((2, H, W), -7., device="cuda")
            s = torch.cuda.Stream()
            torch.cuda.synchronize()
            if mixed:
                ctx.render_frames([_lib.make_frame(slot, p, W, H, o[0].data_ptr(), o[1].data_ptr())],
                                  filter=filt, stream=s.cuda_stream)
            else:
                ctx.render_slot(slot, p, _lib.METHOD_MAX_PROJECT, W, H, o[0].data_ptr(),
                                o[1].data_ptr(), stream=s.cuda_stream)
            s.synchronize()
            outs.append(o.cpu().numpy())
        ctx.close()
        assert (outs[1][0] == .5).all(), (a, b)
        np.testing.assert_array_equal(outs[0], outs[1], err_msg="box -%r %r" % (a, b))
