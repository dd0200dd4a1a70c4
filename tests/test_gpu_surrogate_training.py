"""The training loop and the held-out loss, whose batches torch gathers on its
own stream, against the same batches gathered and synchronised one by one
(bit for bit: every sum runs in a fixed order)."""
import math

import numpy as np
import pytest
import torch

from xbeach_gpu_amd import sur_train
from xbeach_gpu_amd.surrogate import Surrogate

pytestmark = pytest.mark.gpu


def test_loop_equals_synchronised_batches(need_gpu):
    S, H, W, batch, epochs, lr, lr_final = 31, 64, 256, 6, 2, 1e-3, 1e-4
    g = torch.Generator().manual_seed(8)
    X = torch.randn(S, H, W, 8, generator=g).to(torch.bfloat16).cuda()
    T = torch.randn(S, H, W, 5, generator=g).to(torch.bfloat16).cuda()
    torch.cuda.synchronize()
    sur, hist, _, held, nstep = sur_train.train(X, T, epochs, batch, lr, seed=3, log=lambda m: None, lr_final=lr_final)
    got = sur.get_params()
    sur.close()

    g = torch.Generator().manual_seed(3)
    perm = torch.randperm(S, generator=g)
    ntr = int(0.8 * S)
    s = Surrogate(batch, H, W, seed=3)

    def pick(i):
        xb, tb = X[i.cuda()].contiguous(), T[i.cuda()].contiguous()
        torch.cuda.synchronize()
        return xb, tb

    ref, k, total = [], 0, epochs * (ntr // batch)
    for _ in range(epochs):
        order = perm[:ntr][torch.randperm(ntr, generator=g)]
        losses = []
        for j in range(0, ntr - batch + 1, batch):
            xb, tb = pick(order[j:j + batch])
            rate = lr_final + 0.5 * (lr - lr_final) * (1.0 + math.cos(math.pi * k / (total - 1)))
            losses.append(s.train_step(xb.data_ptr(), tb.data_ptr(), batch, rate))
            s.sync()
            k += 1
        ref.append(sum(losses) / len(losses))
    tot, te = 0.0, perm[ntr:]
    for j in range(0, len(te), batch):
        xb, tb = pick(te[j:j + batch])
        tot += s.loss(xb.data_ptr(), tb.data_ptr(), len(xb)) * len(xb)
    assert nstep == k and hist == ref and held == tot / len(te)
    assert np.array_equal(got, s.get_params())
    s.close()
