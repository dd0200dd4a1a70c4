"""The network's fused passes against the same network run pass by pass: each
convolution, data and weight gradient through its layer entry point, the
pooling, upsampling, concatenation, activation masks and the output head as
plain torch operations with every stored tensor rounded to BF16.

Sizes: one tile row per level, tiles of one and of four 16-pixel blocks per
wave at the coarsest level, 32- and 64-pixel rows there.

Tolerances.  The tensors between the passes are BF16 and rounded alike on
both sides, so they are equal bit for bit and only sums in FP32 differ, by
their order: the head's 32 products (32 x 2^-24 of the sum of their sizes),
and the weight and bias gradients, sums of up to n H W products whose
rounding errors grow like the square root of their number: at most
sqrt(n H W) x 2^-24 x 8 of the largest possible sum in the layer, taken as
the 2-norm of the layer's gradient with a floor for layers of small gradient.
"""
import numpy as np
import pytest
import torch

from xbeach_gpu_amd import lib
from xbeach_gpu_amd.surrogate import LAYERS, Surrogate, param_layout

pytestmark = pytest.mark.gpu


def rnd(*shape, g):
    return torch.randn(*shape, generator=g)


class Passes:
    """The network from the layer entry points and torch."""

    def __init__(self, P):
        lay, _ = param_layout()
        self.L = lib()
        self.w, self.b = [], []
        for w, b, cin, cout, taps, _ in lay:
            self.w.append(torch.as_tensor(P[w:b]).reshape(taps, cout, cin).to(torch.bfloat16).contiguous().cuda())
            self.b.append(torch.as_tensor(P[b:b + cout]).float().contiguous().cuda())
        hd = lay[17]
        self.wh = torch.as_tensor(P[hd[0]:hd[1]]).reshape(5, 32).float().cuda()
        self.gw, self.gb = {}, {}

    def conv(self, l, X):
        n, H, W, cin = X.shape
        _, cout, taps, relu = LAYERS[l]
        Y = torch.empty(n, H, W, cout, dtype=torch.bfloat16, device="cuda")
        X = X.contiguous()
        torch.cuda.synchronize()
        assert self.L.xbg_sur_conv_fwd(X.data_ptr(), self.w[l].data_ptr(), self.b[l].data_ptr(), Y.data_ptr(), n, H, W,
                                       cin, cout, taps, relu) == 0
        return Y

    def back(self, l, X, g, need_dx=True):
        """weight and bias gradients of layer l, and its data gradient"""
        n, H, W, cin = X.shape
        _, cout, taps, _ = LAYERS[l]
        X, g = X.contiguous(), g.contiguous()
        dW = torch.empty(taps, cout, cin, device="cuda")
        db = torch.empty(cout, device="cuda")
        dX = torch.empty(n, H, W, cin, dtype=torch.bfloat16, device="cuda")
        torch.cuda.synchronize()
        assert self.L.xbg_sur_conv_wgrad(X.data_ptr(), g.data_ptr(), dW.data_ptr(), db.data_ptr(), n, H, W, cin, cout,
                                         taps) == 0
        self.gw[l], self.gb[l] = dW, db
        if need_dx:
            assert self.L.xbg_sur_conv_dgrad(g.data_ptr(), self.w[l].data_ptr(), dX.data_ptr(), n, H, W, cin, cout,
                                             taps) == 0
            return dX


def quads(x):
    return x[:, ::2, ::2].float(), x[:, ::2, 1::2].float(), x[:, 1::2, ::2].float(), x[:, 1::2, 1::2].float()


def pool(x):
    a, b, c, d = quads(x)
    return (0.25 * (((a + b) + c) + d)).to(torch.bfloat16)


def up(x):
    return x.repeat_interleave(2, 1).repeat_interleave(2, 2)


def up_back(g):
    a, b, c, d = quads(g)
    return (((a + b) + c) + d).to(torch.bfloat16)


def mask(g, y):
    return torch.where(y.float() > 0, g, torch.zeros_like(g))


def unpool_add(gp, skip):
    return (0.25 * up(gp).float() + skip.float()).to(torch.bfloat16)


@pytest.mark.parametrize("n,H,W", [(1, 16, 256), (2, 48, 256), (1, 64, 256), (2, 16, 512), (1, 32, 1024)])
def test_fused_network_equals_its_passes(need_gpu, n, H, W):
    s = Surrogate(n, H, W, seed=n + H)
    g = torch.Generator().manual_seed(H + W)
    P = s.get_params() + 0.05 * np.random.default_rng(1).standard_normal(s.nparams).astype(np.float32)
    s.set_params(P)
    x8 = rnd(n, H, W, 8, g=g).to(torch.bfloat16)
    x8[..., 7] = 0
    x8, t = x8.cuda(), rnd(n, H, W, 5, g=g).to(torch.bfloat16).cuda()
    y = torch.empty(n, H, W, 5, device="cuda")
    torch.cuda.synchronize()
    s.forward(x8.data_ptr(), n, y.data_ptr())
    loss = s.backward(x8.data_ptr(), t.data_ptr(), n)
    G = s.grads()
    s.close()

    p = Passes(P)
    x32 = torch.zeros(n, H, W, 32, dtype=torch.bfloat16, device="cuda")
    x32[..., :8] = x8
    e0a = p.conv(0, x32)
    e0 = p.conv(1, e0a)
    p1 = pool(e0)
    e1a = p.conv(2, p1)
    e1 = p.conv(3, e1a)
    p2 = pool(e1)
    e2a = p.conv(4, p2)
    e2 = p.conv(5, e2a)
    p3 = pool(e2)
    b3a = p.conv(6, p3)
    b3 = p.conv(7, b3a)
    c2 = torch.cat([up(p.conv(8, b3)), e2], -1)
    d2a = p.conv(9, c2)
    d2 = p.conv(10, d2a)
    c1 = torch.cat([up(p.conv(11, d2)), e1], -1)
    d1a = p.conv(12, c1)
    d1 = p.conv(13, d1a)
    c0 = torch.cat([up(p.conv(14, d1)), e0], -1)
    d0a = p.conv(15, c0)
    d0 = p.conv(16, d0a)
    d0f = d0.float().reshape(-1, 32)
    yr = (d0f @ p.wh.T + p.b[17]).reshape(n, H, W, 5)
    tol = 64 * 2.0 ** -24 * (d0f.abs() @ p.wh.abs().T + p.b[17].abs()).max().item()
    assert (y - yr).abs().max().item() <= tol
    assert loss == pytest.approx(((y - t.float()) ** 2).double().mean().item(), rel=1e-5)

    # backward on the library's own outputs
    # an IEEE quotient: torch divides by a plain number through its reciprocal
    gy = 2.0 * (y - t.float()) / torch.full_like(y, y.numel())
    gd0 = torch.zeros(n, H, W, 32, device="cuda")
    for k in range(5):
        gd0 += gy[..., k:k + 1] * p.wh[k]
    g = mask(gd0.to(torch.bfloat16), d0)
    gw17, gb17 = gy.reshape(-1, 5).T.double() @ d0f.double(), gy.reshape(-1, 5).double().sum(0)
    g = mask(p.back(16, d0a, g), d0a)
    gc = p.back(15, c0, g)
    ge0, g = gc[..., 32:], up_back(gc[..., :32])
    g = mask(p.back(14, d1, g), d1)
    g = mask(p.back(13, d1a, g), d1a)
    gc = p.back(12, c1, g)
    ge1, g = gc[..., 64:], up_back(gc[..., :64])
    g = mask(p.back(11, d2, g), d2)
    g = mask(p.back(10, d2a, g), d2a)
    gc = p.back(9, c2, g)
    ge2, g = gc[..., 128:], up_back(gc[..., :128])
    g = mask(p.back(8, b3, g), b3)
    g = mask(p.back(7, b3a, g), b3a)
    g = mask(unpool_add(p.back(6, p3, g), ge2), e2)
    g = mask(p.back(5, e2a, g), e2a)
    g = mask(unpool_add(p.back(4, p2, g), ge1), e1)
    g = mask(p.back(3, e1a, g), e1a)
    g = mask(unpool_add(p.back(2, p1, g), ge0), e0)
    g = mask(p.back(1, e0a, g), e0a)
    p.back(0, x32, g, need_dx=False)
    lay, _ = param_layout()
    rel = 8 * (n * H * W) ** 0.5 * 2.0 ** -24
    for l, (w, b, cin, cout, taps, _) in enumerate(lay):
        gw = torch.as_tensor(G[w:b]).reshape(taps, cout, cin).double()
        gb = torch.as_tensor(G[b:b + cout]).double()
        rw, rb = (gw17.cpu().reshape(1, 5, 32), gb17.cpu()) if l == 17 else (p.gw[l].cpu().double(), p.gb[l].cpu().double())
        for what, a, r in (("weights", gw, rw), ("bias", gb, rb)):
            err, scale = (a - r).norm().item(), r.norm().item()
            assert scale > 0 and err <= rel * scale, (l, what, err, scale)


@pytest.mark.parametrize("n,H,W,cin,cout,taps", [(1, 5, 40, 32, 32, 9), (1, 7, 96, 64, 32, 9), (2, 3, 160, 32, 64, 1),
                                                 (1, 9, 33, 64, 64, 9), (3, 1, 64, 32, 32, 9), (1, 33, 64, 64, 64, 9),
                                                 (2, 19, 128, 32, 64, 9), (1, 2, 32, 32, 32, 1)])
def test_weight_gradient_at_the_edges_of_its_stages(need_gpu, n, H, W, cin, cout, taps):
    """Strips and row stages that do not divide, against torch on the CPU
    (1e-5: FP32 sums in another order, as for the other weight gradients)."""
    import torch.nn.functional as F

    k = 3 if taps == 9 else 1
    g = torch.Generator().manual_seed(H * W + cin)
    X, dZ = rnd(n, H, W, cin, g=g).to(torch.bfloat16), rnd(n, H, W, cout, g=g).to(torch.bfloat16)
    Xd, dZd = X.cuda(), dZ.cuda()
    dW, db = torch.empty(taps, cout, cin, device="cuda"), torch.empty(cout, device="cuda")
    torch.cuda.synchronize()
    assert lib().xbg_sur_conv_wgrad(Xd.data_ptr(), dZd.data_ptr(), dW.data_ptr(), db.data_ptr(), n, H, W, cin, cout,
                                    taps) == 0
    w = torch.zeros(cout, cin, k, k, requires_grad=True)
    b = torch.zeros(cout, requires_grad=True)
    F.conv2d(X.float().permute(0, 3, 1, 2), w, b, padding=k // 2).backward(dZ.float().permute(0, 3, 1, 2))
    for a, r in ((dW.cpu().reshape(k, k, cout, cin).permute(2, 3, 0, 1), w.grad), (db.cpu(), b.grad)):
        assert (a - r).abs().max().item() <= 1e-5 * r.abs().max().item()


def test_inputs_at_any_element_address(need_gpu):
    """Inputs and targets that start 2 bytes into an allocation give the same
    loss, outputs and gradients (the kernels read 8 and 16 bytes at a time)."""
    n, H, W = 1, 16, 256
    s = Surrogate(n, H, W, seed=2)
    g = torch.Generator().manual_seed(5)
    x, t = rnd(n * H * W * 8, g=g).to(torch.bfloat16), rnd(n * H * W * 5, g=g).to(torch.bfloat16)
    got = []
    for shift in (0, 1):
        xd = torch.empty(x.numel() + 1, dtype=torch.bfloat16, device="cuda")[shift:shift + x.numel()].copy_(x)
        td = torch.empty(t.numel() + 1, dtype=torch.bfloat16, device="cuda")[shift:shift + t.numel()].copy_(t)
        y = torch.empty(n, H, W, 5, device="cuda")
        torch.cuda.synchronize()
        s.forward(xd.data_ptr(), n, y.data_ptr())
        got.append((s.backward(xd.data_ptr(), td.data_ptr(), n), y.cpu(), s.grads()))
    s.close()
    assert got[0][0] == got[1][0] and torch.equal(got[0][1], got[1][1]) and np.array_equal(got[0][2], got[1][2])
