"""Saved tensors of posteriors and samples that come back from hooks on another device,
in another type or layout, and the bound on what posteriors hold until their backward.
The compared gradients come from the same kernels on the same
inputs: equal bit for bit."""
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


def _samples(mean, cov, z):
    return B.GPyTorchPosterior(mean, cov).rsample_from_base_samples(
        torch.Size([16]), z).squeeze(-1)


@pytest.mark.parametrize("how", ["cpu", "single", "cpu single", "strided"])
@pytest.mark.parametrize("shared", [True, False])
def test_saved_base_samples_may_come_back_as_other_tensors(how, shared):
    g = torch.Generator().manual_seed(2)
    A = torch.randn(3, 4, 4, generator=g, dtype=torch.float64)
    cov = (A @ A.transpose(-1, -2) + 4 * torch.eye(4, dtype=torch.float64)).to(DEV)
    mean = torch.randn(3, 4, generator=g, dtype=torch.float64).to(DEV)
    # exact in single precision
    z = torch.randn(16, 3, 4, generator=g, dtype=torch.float32).double().to(DEV)
    w = torch.randn(16, 3, 4, generator=g, dtype=torch.float64).to(DEV)
    if shared:
        z = z[:, :1].expand(16, 3, 4)
    mean.requires_grad_(True)
    cov.requires_grad_(True)
    want = torch.autograd.grad(_samples(mean, cov, z), (mean, cov), w)

    def pack(t):
        if t.shape != z.shape:
            return t
        t = t.cpu() if "cpu" in how else t
        if how == "strided":
            return t.permute(2, 0, 1).contiguous().permute(1, 2, 0)
        return t.float() if "single" in how else t

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t):
        y = _samples(mean, cov, z)
    got = torch.autograd.grad(y, (mean, cov), w)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("kept", [True, False])
def test_saved_posterior_tensors_may_come_back_in_another_type(monkeypatch, kept):
    if not kept:
        monkeypatch.setattr(G, "KEEP_BYTES", 0)
    gp = _model()
    # exact in single precision
    X = torch.rand(5, 2, 3, generator=torch.Generator().manual_seed(2)).double().to(DEV)
    X.requires_grad_(True)

    def grad():
        post = gp.posterior(X)
        return post.covariance_matrix.square().sum() + post.mean.sum()

    (want,) = torch.autograd.grad(grad(), X)

    def pack(t):
        if t.dtype == torch.uint8:
            return t.short().cpu()
        return t.float().cpu() if t.shape == X.shape else t

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t):
        loss = grad()
    assert torch.equal(torch.autograd.grad(loss, X)[0], want)


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
    for _ in range(2):  # what the first pass held is free again in the second
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
