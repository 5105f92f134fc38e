"""A posterior's backward on a stream of its own reads the prediction cache of its forward
pass: the cache's memory is not given out again before it is done, also when the graph
held the last reference.  The compared gradients come from the same kernels on the same
inputs: equal bit for bit."""
import pytest
import torch

import botorch_amd as B
from botorch_amd import gp as G

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("kept", [True, False])
def test_a_dropped_cache_outlives_the_backward_on_another_stream(monkeypatch, kept):
    if not kept:
        monkeypatch.setattr(G, "KEEP_BYTES", 0)
    g = torch.Generator().manual_seed(5)
    X = torch.rand(300, 3, generator=g, dtype=torch.float64)
    gp = B.SingleTaskGP(X.to(DEV), torch.sin(5 * X).sum(-1, keepdim=True).to(DEV))
    Xq = torch.rand(4, 3, 3, generator=g, dtype=torch.float64).to(DEV).requires_grad_(True)
    ls = gp.covar_module.lengthscale.detach().clone()

    def loss_of():
        post = gp.posterior(Xq)
        return post.covariance_matrix.square().sum() + post.mean.sum()

    (want,) = torch.autograd.grad(loss_of(), Xq)
    sizes = [t.shape for t in gp.prediction_cache().values() if torch.is_tensor(t)]
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        loss = loss_of()
    gp.covar_module.lengthscale = 3.0 * ls
    gp.prediction_cache()  # the graph holds the old cache alone now
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        torch.cuda._sleep(50_000_000)  # tens of milliseconds ahead of the backward
        (got,) = torch.autograd.grad(loss, Xq)
        del loss
    # what memory the allocator gives out now is overwritten while the side stream sleeps
    fills = [torch.full(size, float("nan"), dtype=torch.float64, device=DEV)
             for size in sizes for _ in range(3)]
    torch.cuda.current_stream().synchronize()
    side.synchronize()
    assert torch.equal(got, want) and len(fills) > 0
