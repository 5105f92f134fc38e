"""What posteriors that wait for their backward hold: with saved-tensor hooks, tensors
that come back on another device or in another type; and no more than KEEP_BYTES in all.
The compared gradients come from the same kernels on the same inputs: equal bit for bit."""
import pytest
import torch

import botorch_amd as B
from botorch_amd import gp as G

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _model(n=100, d=3):
    g = torch.Generator().manual_seed(5)
    X = torch.rand(n, d, generator=g, dtype=torch.float64)
    Y = torch.sin(5 * X).sum(-1, keepdim=True)
    return B.SingleTaskGP(X.to(DEV), Y.to(DEV))


def test_many_live_posteriors_hold_a_bounded_amount(monkeypatch):
    gp = _model()
    g = torch.Generator().manual_seed(1)
    Xs = [torch.rand(64, 4, 3, generator=g, dtype=torch.float64).to(DEV) for _ in range(20)]
    gp.prediction_cache()
    alone = []
    for X in Xs:
        X.requires_grad_(True)
        post = gp.posterior(X)
        (dx,) = torch.autograd.grad(post.covariance_matrix.square().sum(), X)
        alone.append(dx)
    per = 256 * 128 * 8  # rows x n_pad doubles of V
    limit = 4 * per
    monkeypatch.setattr(G, "KEEP_BYTES", limit)
    for _ in range(2):  # what the first round held is free again in the second
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        posts = [gp.posterior(X) for X in Xs]
        held = torch.cuda.memory_allocated() - before
        outputs = len(Xs) * (64 * 4 * 4 + 64 * 4) * 8
        assert per < held < limit + outputs + len(Xs) * 64 * 1024, held
        loss = sum(p.covariance_matrix.square().sum() for p in posts)
        together = torch.autograd.grad(loss, Xs)
        assert all(torch.equal(a, b) for a, b in zip(alone, together))
        del posts, loss, together
