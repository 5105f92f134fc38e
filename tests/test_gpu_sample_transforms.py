"""Posterior samples under the other ways of differentiating and mapping them: a second
derivative through the mean, forward mode, vmap and batched gradients over the mean.

The samples are mean + L z, linear in the mean: every expected value is formed from the
samples themselves, up to one rounding per operation (1e-13 of values of order 10)."""
import pytest
import torch
import torch.autograd.forward_ad as fwAD

import botorch_amd as B

pytestmark = pytest.mark.gpu
DEV = "cuda"
NB, M, S = 3, 4, 16
SHAPE = torch.Size([S])


def _parts():
    g = torch.Generator().manual_seed(2)
    A = torch.randn(NB, M, M, generator=g, dtype=torch.float64)
    cov = (A @ A.transpose(-1, -2) + M * torch.eye(M, dtype=torch.float64)).to(DEV)
    mean = torch.randn(NB, M, generator=g, dtype=torch.float64).to(DEV)
    z = torch.randn(S, NB, M, generator=g, dtype=torch.float64).to(DEV)
    w = torch.randn(S, NB, M, generator=g, dtype=torch.float64).to(DEV)
    return mean, cov, z, w


def _samples(mean, cov, z):
    return B.GPyTorchPosterior(mean, cov).rsample_from_base_samples(SHAPE, z).squeeze(-1)


@pytest.mark.parametrize("cov_grad", [False, True])
def test_second_derivative_in_the_mean(cov_grad):
    mean, cov, z, _ = _parts()
    mean.requires_grad_(True)
    cov.requires_grad_(cov_grad)
    y = _samples(mean, cov, z)
    (g,) = torch.autograd.grad((y ** 3).sum(), mean, create_graph=True)
    assert (g - 3 * y.square().sum(0)).abs().max() < 1e-13 * g.abs().max()
    (h,) = torch.autograd.grad(g.sum(), mean)
    want = 6 * y.detach().sum(0)
    assert (h - want).abs().max() < 1e-13 * y.abs().sum(0).max() * 6


def test_forward_mode_in_the_mean():
    mean, cov, z, _ = _parts()
    t = torch.randn_like(mean)
    with fwAD.dual_level():
        y = _samples(fwAD.make_dual(mean, t), cov, z)
        primal, tangent = fwAD.unpack_dual(y)
        assert tangent is not None
        assert torch.equal(tangent, t.expand(S, NB, M))
        assert (primal - _samples(mean, cov, z)).abs().max() < 1e-13 * primal.abs().max()


def test_vmap_over_the_mean():
    mean, cov, z, _ = _parts()
    means = torch.stack([mean, 2 * mean, -mean])
    y = torch.func.vmap(lambda mu: _samples(mu, cov, z))(means)
    for mu, ys in zip(means, y):
        assert (ys - _samples(mu, cov, z)).abs().max() < 1e-13 * ys.abs().max()


def test_batched_gradients_of_the_mean():
    mean, cov, z, w = _parts()
    mean.requires_grad_(True)
    ws = torch.stack([w, 2 * w])
    (g,) = torch.autograd.grad(_samples(mean, cov, z), mean, ws, is_grads_batched=True)
    assert (g - ws.sum(1)).abs().max() < 1e-13 * ws.abs().sum(1).max()
