"""Device bytes of a resident volume: what a slot reports is what it takes -- voxels, window
grid and brick keys -- and what the render server reserves for it."""
import numpy as np
import pytest

from spimagine_amd import _lib
from spimagine_amd.serving import RenderServer, Request, device_bytes


def test_bytes_of_windows_and_bricks():
    # 66 x 130 x 136 uint16 padded (rows of 16 bytes), 17 x 33 x 33 windows, 9 x 17 x 17 bricks
    pad, win, bricks = 66 * 130 * 136 * 2, 17 * 33 * 33 * 2, 9 * 17 * 17 + 2
    up = lambda n: (n + 255) // 256 * 256  # noqa: E731
    assert _lib.Context.volume_bytes((64, 128, 128), np.uint16) == up(pad) + 2 * up(win) + 8 * bricks
    big = (512, 2048, 2048)
    assert _lib.Context.volume_bytes(big, np.uint16) > device_bytes(big, np.uint16) * 65 // 64


class Slots(object):
    """A context that only counts (no GPU)."""
    volume_bytes = staticmethod(_lib.Context.volume_bytes)

    def __init__(self):
        self.slots = {}

    def volume_add(self, data):
        self.slots[len(self.slots) + 1] = data
        return len(self.slots)

    def volume_info(self, slot):
        d = self.slots[slot]
        return {"dtype": 1, "shape": d.shape, "bytes": self.volume_bytes(d.shape, d.dtype)}

    def volume_release(self, slot):
        self.slots[slot] = None

    def close(self):
        pass


def test_server_stays_within_its_budget():
    """Two volumes whose voxels alone fit the budget, but not with their bounds: the second is
    admitted only once the first can go."""
    vol = np.zeros((62, 62, 62), np.uint16)
    srv = RenderServer(hbm_budget=2 * device_bytes(vol.shape, vol.dtype) + 1000, workers=0, ctx=Slots())
    for name in "ab":
        srv.register(name, vol)
        srv.submit(Request(name, np.eye(4), np.eye(4), size=(16, 16)))
    first = srv._take_batch()
    assert [r.volume for r, _ in first] == ["a"]
    assert srv._take_batch() is None and srv.resident_bytes <= srv.hbm_budget
    srv.volumes["a"].users -= 1
    assert [r.volume for r, _ in srv._take_batch()] == ["b"]
    assert srv.resident_bytes <= srv.hbm_budget


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.uint16, np.uint8, np.float32])
@pytest.mark.parametrize("shape", [(64, 128, 128), (33, 90, 70), (1, 2, 3), (130, 129, 131)])
def test_a_slot_reports_its_allocations(dtype, shape):
    ctx = _lib.Context(0)
    slot = ctx.volume_add(np.ones(shape, dtype))
    assert ctx.volume_info(slot)["bytes"] == _lib.Context.volume_bytes(shape, dtype)
    if dtype == np.uint16:  # a pair: two channels a voxel, windows, no bricks
        pair = ctx.volume_add_pooled_pair(slot)
        small = tuple((n + 1) // 2 for n in shape)
        bricks = 8 * (int(np.prod([(n + 9) // 8 for n in small])) + 2)
        assert ctx.volume_info(pair)["bytes"] == _lib.Context.volume_bytes(small, np.float32) - bricks
    ctx.set_layout(_lib.LAYOUT_LINEAR)
    lin = ctx.volume_add(np.ones(shape, dtype))
    assert ctx.volume_info(lin)["bytes"] == int(np.prod(shape)) * np.dtype(dtype).itemsize
    ctx.close()

