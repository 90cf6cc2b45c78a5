"""GPU: the weight gradients of every layer against float64 sums of the same operands, and with
an infinite target."""
import numpy as np
import pytest

from spimagine_amd import learned

pytestmark = pytest.mark.gpu


def gradients(params, x, tgt):
    import torch
    net = learned.Net(0, params)
    dx, dt = torch.from_numpy(x).cuda(), torch.from_numpy(tgt).cuda()
    g, sse = net.gradients(dx.data_ptr(), dt.data_ptr(), x.shape[0], x.shape[2], x.shape[3])
    net.close()
    return learned.split_params(g), sse


def uniform_net(w, b):
    flat = learned.init_params(0)
    for k, v in learned.split_params(flat).items():
        v[...] = b if k.endswith(".b") else w
    return flat


# positive weights and activations: every sum of an infinite gradient has one sign
def test_an_infinite_target_leaves_infinite_gradients():
    h, w = 96, 96
    x = np.full((1, 2, h, w), .5, np.float32)
    tgt = np.zeros((1, 2 * h, 2 * w), np.float32)
    tgt[0, 96, 97] = np.inf  # one sub-pixel in the middle: head channel 1
    g, _ = gradients(uniform_net(.01, .1), x, tgt)
    head = np.zeros((9, learned.C, 4), bool)
    head[:, :, 1] = True
    np.testing.assert_array_equal(np.isneginf(g["head.w"]), head)
    assert np.isfinite(g["head.w"][~head]).all()
    np.testing.assert_array_equal(np.isneginf(g["head.b"]), [False, True, False, False])
    for k, v in g.items():
        if not k.startswith("head"):
            assert np.isneginf(v).all(), k


def bf(t):
    import torch
    return t.to(torch.bfloat16).to(torch.float32)


# A network whose layers' operands are known exactly: single taps of powers of two, the coarse
# levels switched off, so that activations and gradients are the input's and the loss's values,
# scaled, rounded to bf16 only where the kernels round them.
@pytest.mark.parametrize("n,h,w", [(1, 40, 72), (3, 64, 96)])
def test_weight_gradients_keep_float32_precision(n, h, w):
    import torch
    F = torch.nn.functional
    C = learned.C
    rng = np.random.default_rng(h)
    flat = np.zeros(learned.param_count(), np.float32)
    p = learned.split_params(flat)
    ch = np.arange(C)
    for name in ("e0", "e0b", "u0", "u0b"):
        p[name + ".w"][4, ch, ch] = 1.
        p[name + ".w"][4, ch, (ch + 1) % C] = 2. ** -6  # a second term: gradients of 16 bits
    p["in.w"][4, ch % 2, ch] = 2. ** -(ch % 3)
    p["head.w"][4, ch, ch % 4] = 2. ** (ch % 3 - 1)
    p["e1.b"][...] = p["u1.b"][...] = -1.  # relu: no coarse level
    x = rng.uniform(.1, 1., (n, 2, h, w)).astype(np.float32)
    tgt = rng.uniform(-1., 1., (n, 2 * h, 2 * w)).astype(np.float32)
    g, _ = gradients(flat, x, tgt)

    def conv(t, wt, back=False):  # few exact terms: any order of sums
        cin, cout = wt.shape[1], wt.shape[2]
        k = torch.from_numpy(wt.reshape(3, 3, cin, cout)).permute(3, 2, 0, 1)
        return (F.conv_transpose2d if back else F.conv2d)(t.double(), k.double(), padding=1).float()

    def check(name, act, grad):
        u = F.unfold(act.double(), 3, padding=1).reshape(n, act.shape[1], 9, h * w)
        dw = torch.einsum("nctp,nop->tco", u, grad.double().reshape(n, -1, h * w)).numpy()
        db = grad.double().sum((0, 2, 3)).numpy()
        for k, want in ((name + ".w", dw), (name + ".b", db)):
            rel = np.linalg.norm(g[k] - want) / np.linalg.norm(want)
            # float32 sums of a full batch of 512^2 frames are off by 5.5e-7 of the norm; two
            # pieces of bf16 instead of three would be off by 1e-5, one by 3e-3
            assert rel <= 2e-6, (k, rel)

    tx = torch.from_numpy(x)
    a0 = bf(F.relu(conv(tx, p["in.w"])))
    e0 = bf(F.relu(conv(a0, p["e0.w"])))
    e0b = bf(F.relu(conv(e0, p["e0b.w"])))
    u0 = bf(F.relu(conv(e0b, p["u0.w"])))
    u0b = bf(F.relu(conv(u0, p["u0b.w"])))
    r = conv(u0b, p["head.w"])
    # the loss's gradient as the kernels see it: the output read back, 2 (y - target) / count
    net = learned.Net(0, flat)
    y = torch.empty((n, 2 * h, 2 * w), device="cuda")
    dx = tx.cuda()
    net.forward(dx.data_ptr(), n, h, w, y.data_ptr())
    net.close()
    torch.cuda.synchronize()
    y = y.cpu().numpy()
    base = F.interpolate(tx[:, :1], scale_factor=2, mode="bilinear", align_corners=False)
    np.testing.assert_allclose(y, (F.pixel_shuffle(r, 2) + base)[:, 0].numpy(), rtol=0, atol=1e-5)
    scale = np.float32(2.) / np.float32(y.size)
    dr = F.pixel_unshuffle(torch.from_numpy(scale * (y - tgt))[:, None], 2)
    check("head", u0b, dr)
    d = conv(dr, p["head.w"], back=True)
    check("u0b", u0, d)  # (every activation is positive)
    d = conv(bf(d), p["u0b.w"], back=True)
    check("u0", e0b, d)
    d = conv(bf(d), p["u0.w"], back=True)
    check("e0b", e0, d)
    d = conv(bf(d), p["e0b.w"], back=True)
    check("e0", a0, d)
    d = conv(bf(d), p["e0.w"], back=True)
    check("in", tx, d)
