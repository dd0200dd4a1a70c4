"""A training step is done with the caller's batch when it returns: buffers
that are refilled right behind the call give the same loss, gradients and
weights as untouched ones (bit for bit: the sums run in a fixed order)."""
import numpy as np
import pytest
import torch

from xbeach_gpu_amd.surrogate import Surrogate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,H,W", [(1, 16, 256), (8, 256, 256)])
def test_batch_refilled_behind_a_training_step(need_gpu, n, H, W):
    g = torch.Generator().manual_seed(H)
    x = torch.randn(n, H, W, 8, generator=g).to(torch.bfloat16).cuda()
    t = torch.randn(n, H, W, 5, generator=g).to(torch.bfloat16).cuda()
    got = []
    for refill in (False, True):
        s = Surrogate(n, H, W, seed=4)
        losses = []
        for _ in range(3):
            xb, tb = x.clone(), t.clone()
            torch.cuda.synchronize()
            losses.append(s.train_step(xb.data_ptr(), tb.data_ptr(), n, 1e-3))
            if refill:
                xb.fill_(100.0)
                tb.fill_(-100.0)
            else:
                s.sync()
        got.append((losses, s.grads(), s.get_params()))
        s.close()
    assert got[0][0] == got[1][0]
    assert np.array_equal(got[0][1], got[1][1]) and np.array_equal(got[0][2], got[1][2])
