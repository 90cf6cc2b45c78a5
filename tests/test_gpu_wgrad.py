"""GPU: the network's gradients where the weight-gradient kernels' 32 x 8 tiles are ragged:
against autograd of the float32 reference, and a batch against its images one by one."""
import numpy as np
import pytest

from spimagine_amd import learned
from test_gpu_learned import random_params, ref_forward_t, smooth_inputs

pytestmark = pytest.mark.gpu


def gradients(torch, net, x, tgt):
    dx, dt = torch.from_numpy(x).cuda(), torch.from_numpy(tgt).cuda()
    return net.gradients(dx.data_ptr(), dt.data_ptr(), x.shape[0], x.shape[2], x.shape[3])


# one partial tile at every level; one row of tiles and a rest; a rest in both; many tiles
@pytest.mark.parametrize("n,h,w", [(1, 4, 4), (1, 8, 36), (2, 12, 32), (2, 44, 100), (4, 136, 260)])
def test_gradients_on_ragged_tiles(n, h, w):
    import torch
    rng = np.random.default_rng(h + w)
    params = random_params(3)
    x = smooth_inputs(rng, n, h, w)
    tgt = rng.uniform(0, 1, (n, 2 * h, 2 * w)).astype(np.float32)
    net = learned.Net(0, params)
    g, sse = gradients(torch, net, x, tgt)
    # images one by one: the mean over n (a power of two) scales every loss term exactly, so
    # only the order of float32 additions differs (1e-6 of the norm measured on such sums)
    parts = [gradients(torch, net, x[k:k + 1].copy(), tgt[k:k + 1].copy()) for k in range(n)]
    net.close()
    mean = np.mean([p[0].astype(np.float64) for p in parts], axis=0)
    assert np.linalg.norm(g - mean) <= 1e-5 * np.linalg.norm(mean)
    assert abs(sse - sum(p[1] for p in parts)) <= 1e-5 * sse
    pt = torch.from_numpy(params.copy()).requires_grad_(True)
    y = ref_forward_t(torch, pt, torch.from_numpy(x))
    (((y - torch.from_numpy(tgt)) ** 2).sum() / y.numel()).backward()
    gr, k = pt.grad.numpy().astype(np.float64), 0
    for name, shape in learned.param_layout():
        m = int(np.prod(shape))
        a, b = g[k:k + m].astype(np.float64), gr[k:k + m]
        k += m
        # bf16 activations and gradients of the layers behind, as in the other gradient test
        cos = a @ b / (np.linalg.norm(a) * np.linalg.norm(b) + 1e-30)
        rel = np.linalg.norm(a - b) / (np.linalg.norm(b) + 1e-30)
        assert cos >= .99 and rel <= .1, (name, cos, rel)
