"""The convolutions' gradients at the edges of what their layer entry points
take."""
import numpy as np
import pytest
import torch

from xbeach_gpu_amd import lib

pytestmark = pytest.mark.gpu


def taps_gradient(X, dZ, taps):
    """Weight gradient in 64 bits, summed over the pixels whose tap lies inside."""
    n, H, W, cin = X.shape
    k = 3 if taps == 9 else 1
    X, dZ = X.double().numpy(), dZ.double().numpy()
    out = np.zeros((taps, dZ.shape[3], cin))
    for tap in range(taps):
        oy, ox = tap // k - k // 2, tap % k - k // 2
        ys, xs = slice(max(0, -oy), H - max(0, oy)), slice(max(0, -ox), W - max(0, ox))
        yi, xi = slice(max(0, oy), H - max(0, -oy)), slice(max(0, ox), W - max(0, -ox))
        with np.errstate(invalid="ignore"):
            out[tap] = dZ[:, ys, xs].reshape(-1, dZ.shape[3]).T @ X[:, yi, xi].reshape(-1, cin)
    return out


@pytest.mark.parametrize("n,H,W,cin,cout,taps", [(1, 5, 40, 32, 32, 9), (2, 4, 33, 64, 32, 9), (1, 9, 95, 32, 64, 9),
                                                 (1, 6, 31, 64, 64, 9), (1, 4, 40, 32, 64, 1), (1, 6, 64, 32, 32, 9)])
def test_infinite_inputs_stay_in_their_taps(need_gpu, n, H, W, cin, cout, taps):
    """An infinite input reaches the gradients of the taps that read it and no
    others: pixels past the last column (their gradient is 0) add nothing.
    Finite values as elsewhere (FP32 sums in another order: 1e-5)."""
    g = torch.Generator().manual_seed(W + cout)
    X = torch.randn(n, H, W, cin, generator=g).to(torch.bfloat16)
    dZ = torch.randn(n, H, W, cout, generator=g).to(torch.bfloat16)
    dZ[dZ == 0] = 1.0
    for c, (y, x) in enumerate([(0, W - 1), (H // 2, W - 1), (H - 1, W - 1), (1, W - 2), (2, 0)]):
        X[n - 1, y, x, 3 * c] = float("inf")
    Xd, dZd = X.cuda(), dZ.cuda()
    dW, db = torch.empty(taps, cout, cin, device="cuda"), torch.empty(cout, device="cuda")
    torch.cuda.synchronize()
    assert lib().xbg_sur_conv_wgrad(Xd.data_ptr(), dZd.data_ptr(), dW.data_ptr(), db.data_ptr(), n, H, W, cin, cout,
                                    taps) == 0
    got, ref = dW.cpu().double().numpy(), taps_gradient(X, dZ, taps)
    fin = np.isfinite(ref)
    assert fin.any() and (~fin).any() and not np.isnan(ref).any()
    assert np.array_equal(got[~fin], ref[~fin])
    assert np.abs(got[fin] - ref[fin]).max() <= 1e-5 * np.abs(ref[fin]).max()


@pytest.mark.parametrize("cin,cout,taps,rc", [(4096, 4096, 1, 0), (448, 4160, 9, 0), (4096, 4128, 1, -1)])
def test_largest_weight_gradient(need_gpu, cin, cout, taps, rc):
    """Layers of up to 2^24 weights are taken, larger ones are refused."""
    n, H, W = 1, 2, 32
    g = torch.Generator().manual_seed(cout)
    X = torch.randn(n, H, W, cin, generator=g).to(torch.bfloat16)
    dZ = torch.randn(n, H, W, cout, generator=g).to(torch.bfloat16)
    Xd, dZd = X.cuda(), dZ.cuda()
    dW, db = torch.empty(taps, cout, cin, device="cuda"), torch.empty(cout, device="cuda")
    torch.cuda.synchronize()
    got = lib().xbg_sur_conv_wgrad(Xd.data_ptr(), dZd.data_ptr(), dW.data_ptr(), db.data_ptr(), n, H, W, cin, cout, taps)
    assert (got == 0) == (rc == 0)
    if rc == 0:
        for a, r in ((dW.cpu().double().numpy(), taps_gradient(X, dZ, taps)),
                     (db.cpu().double().numpy(), dZ.double().numpy().reshape(-1, cout).sum(0))):
            assert np.abs(a - r).max() <= 1e-5 * np.abs(r).max()


def test_data_gradient_of_more_than_2_31_weights(need_gpu):
    """The flipped weights are indexed beyond 2^31: a few weights set, products
    and sums of small integers, so exact."""
    n, H, W, cin, cout, taps = 1, 2, 32, 15456, 15456, 9
    if torch.cuda.mem_get_info()[0] < 12 << 30:
        pytest.skip("needs 12 GB")
    rng = np.random.default_rng(5)
    Wt = torch.zeros(taps * cout * cin, dtype=torch.bfloat16, device="cuda")
    assert Wt.numel() > 1 << 31
    at = np.concatenate([rng.integers(0, Wt.numel(), 200), rng.integers(1 << 31, Wt.numel(), 50),
                         [0, (1 << 31) - 1, 1 << 31, Wt.numel() - 1]])
    at = np.unique(at)
    val = rng.integers(1, 5, at.size)
    Wt[torch.as_tensor(at).cuda()] = torch.as_tensor(val).to(torch.bfloat16).cuda()
    dZ = rng.integers(-3, 4, (H, W, cout))
    dZd = torch.as_tensor(dZ).to(torch.bfloat16).cuda()
    dX = torch.full((H, W, cin), float("nan"), dtype=torch.bfloat16, device="cuda")
    torch.cuda.synchronize()
    assert lib().xbg_sur_conv_dgrad(dZd.data_ptr(), Wt.data_ptr(), dX.data_ptr(), n, H, W, cin, cout, taps) == 0
    ref = np.zeros((H + 2, W + 2, cin))
    for i, v in zip(at, val):
        tap, co, ci = i // (cout * cin), i // cin % cout, i % cin
        ref[tap // 3:tap // 3 + H, tap % 3:tap % 3 + W, ci] += v * dZ[:, :, co]
    assert np.array_equal(dX.cpu().double().numpy(), ref[1:-1, 1:-1])
