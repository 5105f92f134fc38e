"""Posterior moments and their adjoint over both row layouts (packed rows up to 16
points per batch element, rows padded to 64 above) at the edges of their tiles,
against autograd through the FP64 oracle.

Tolerance: the oracle forms distances by the norm expansion and solves with
triangular solves where the library multiplies by L^-1, so the two differ by
rounding amplified by cond(K) <= (n s + noise) / noise = 200 / 1e-2 = 2e4: a few
1e-12 relative to the largest entry, and one order more for the adjoint.  1e-10."""
import pytest
import torch

import botorch_amd as B
from oracle import gp_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _pair(n, d, kind):
    g = torch.Generator().manual_seed(n + d)
    X = torch.rand(n, d, generator=g, dtype=torch.float64)
    Y = torch.sin(3 * X).sum(-1, keepdim=True)
    ls = 0.3 + torch.rand(d, generator=g, dtype=torch.float64)
    base = B.MaternKernel(ard_num_dims=d) if kind == O.MATERN52 else B.RBFKernel(ard_num_dims=d)
    base.lengthscale = ls
    lik = B.GaussianLikelihood()
    lik.noise = 1e-2
    covar = B.ScaleKernel(base)
    covar.outputscale = 1.0
    gp = B.SingleTaskGP(X.to(DEV), Y.to(DEV), likelihood=lik, covar_module=covar)
    return gp, O.OracleGP(X, Y, kind, ls, 1.0, 1e-2)


@pytest.mark.parametrize("n,d,batch,mq,kind", [
    (2, 1, 1, 1, O.RBF), (5, 4, 130, 1, O.MATERN52), (127, 5, 3, 2, O.RBF),
    (128, 8, 43, 3, O.MATERN52), (129, 9, 7, 5, O.RBF), (200, 12, 16, 8, O.MATERN52),
    (150, 13, 2, 9, O.RBF), (100, 16, 9, 15, O.MATERN52), (100, 17, 9, 16, O.RBF),
    (100, 21, 2, 17, O.MATERN52), (190, 28, 2, 64, O.RBF), (190, 32, 1, 65, O.MATERN52),
    (70, 3, 3, 128, O.MATERN52), (200, 6, 1, 193, O.RBF)])
def test_posterior_layouts_match_oracle(n, d, batch, mq, kind):
    print(f"[case] n={n} d={d} batch={batch} mq={mq} kind={kind}", flush=True)
    gp, orc = _pair(n, d, kind)
    g = torch.Generator().manual_seed(mq)
    X = torch.rand(batch, mq, d, generator=g, dtype=torch.float64)
    X[0, 0] = orc.train_X[0]  # a query on a training point
    wm = torch.randn(batch, mq, generator=g, dtype=torch.float64)
    wc = torch.randn(batch, mq, mq, generator=g, dtype=torch.float64)
    Xr = X.clone().requires_grad_(True)
    m_r, c_r = orc.posterior(Xr)
    for wcov in (wc, None):  # with the covariance's adjoint and the mean's alone
        Xd = X.to(DEV).requires_grad_(True)
        post = gp.posterior(Xd)
        loss = (post.mean.squeeze(-1) * wm.to(DEV)).sum()
        ref = (m_r * wm).sum()
        if wcov is not None:
            loss = loss + (post.covariance_matrix * wcov.to(DEV)).sum()
            ref = ref + (c_r * wcov).sum()
        (gd,) = torch.autograd.grad(loss, Xd)
        (gr,) = torch.autograd.grad(ref, Xr, retain_graph=True)
        scale = max(gr.abs().max().item(), 1e-3)
        assert (gd.cpu() - gr).abs().max().item() < 1e-10 * scale
    assert (post.mean.detach().squeeze(-1).cpu() - m_r.detach()).abs().max() < 1e-10 * max(
        1.0, m_r.abs().max().item())
    cov = post.covariance_matrix.detach()
    assert (cov.cpu() - c_r.detach()).abs().max() < 1e-10 * c_r.abs().max()
    assert torch.equal(cov, cov.transpose(-1, -2))
    with torch.no_grad():
        alone = gp.posterior(X[-1:].to(DEV))
    assert (alone.mean - post.mean[-1:].detach()).abs().max() < 1e-10 * max(
        1.0, m_r.abs().max().item())


def test_posterior_nan_stays_in_its_batch_element():
    gp, _ = _pair(60, 4, O.MATERN52)
    for mq in (3, 20):
        X = torch.rand(5, mq, 4, dtype=torch.float64, device=DEV)
        with torch.no_grad():
            ref = gp.posterior(X).covariance_matrix
            X[2, 1, 0] = float("nan")
            cov = gp.posterior(X).covariance_matrix
        assert torch.isnan(cov[2, 1]).all()
        keep = [0, 1, 3, 4]
        assert torch.equal(cov[keep], ref[keep])


@pytest.mark.parametrize("nb,m,S,shared", [(1, 1, 1, True), (3, 4, 64, True), (5, 7, 33, False),
                                           (2, 16, 300, True), (2, 17, 20, True)])
def test_samples_and_their_gradient(nb, m, S, shared):
    """Samples over the packed kernel (m <= 16) and the GEMM above, with base samples
    shared by the batch (an expanded view) or one set each, against torch: sums of at
    most max(m, S) products, 1e-12 of the largest entry."""
    g = torch.Generator().manual_seed(m + S)
    A = torch.randn(nb, m, m, generator=g, dtype=torch.float64)
    cov = (A @ A.transpose(-1, -2) + m * torch.eye(m, dtype=torch.float64)).to(DEV)
    mean = torch.randn(nb, m, generator=g, dtype=torch.float64).to(DEV)
    z = torch.randn(S, 1 if shared else nb, m, generator=g, dtype=torch.float64).to(DEV)
    w = torch.randn(S, nb, m, generator=g, dtype=torch.float64).to(DEV)
    args = [mean.clone().requires_grad_(True), cov.clone().requires_grad_(True)]
    post = B.GPyTorchPosterior(*args)
    out = post.rsample_from_base_samples(torch.Size([S]), z.expand(S, nb, m))
    got = torch.autograd.grad(out.squeeze(-1), args, w)
    ref_args = [mean.cpu().requires_grad_(True), cov.cpu().requires_grad_(True)]
    L = torch.linalg.cholesky(ref_args[1])
    ref = ref_args[0] + torch.stack([(L * v.unsqueeze(-2)).sum(-1)
                                     for v in z.cpu().expand(S, nb, m)])
    want = torch.autograd.grad(ref, ref_args, w.cpu())
    for x, y in zip([out.detach().squeeze(-1), *got], [ref.detach(), *want]):
        assert x.shape == y.shape
        assert (x.cpu() - y).abs().max() < 1e-12 * y.abs().max() * max(m, S)
    with torch.no_grad():
        plain = B.GPyTorchPosterior(mean, cov).rsample_from_base_samples(
            torch.Size([S]), z.expand(S, nb, m))
    assert torch.equal(plain, out.detach())


def test_posterior_adjoint_kept_and_recomputed_agree(monkeypatch):
    """The adjoint from the moments' own buffer equals the one that forms K_x and V
    again (above KEEP_BYTES) bit for bit, and belongs to the hyperparameters of the
    forward pass."""
    from botorch_amd import gp as G
    model, _ = _pair(150, 5, O.MATERN52)
    for mq in (3, 40):
        X = torch.rand(4, mq, 5, dtype=torch.float64, device=DEV, requires_grad=True)
        grads = []
        for limit in (G.KEEP_BYTES, 0):
            monkeypatch.setattr(G, "KEEP_BYTES", limit)
            post = model.posterior(X)
            loss = post.mean.sum() + post.covariance_matrix.square().sum()
            if not limit:
                noise = model.likelihood.noise.detach().clone()
                model.likelihood.noise = 0.5
            grads.append(torch.autograd.grad(loss, X)[0])
        model.likelihood.noise = noise
        monkeypatch.undo()
        assert torch.equal(*grads)


@pytest.mark.parametrize("batch,mq", [(191, 17), (192, 17), (63, 97), (64, 97), (1, 1500)])
def test_posterior_joint_tiles_both_sides_of_their_rule(batch, mq):
    # 2 ceil(mq / 128) (ceil(mq / 128) + 1) batch against 3 x 256 CUs: 32 x 32 tiles of
    # V V^T below, 128 x 64 above
    print(f"[case] batch={batch} mq={mq}", flush=True)
    gp, orc = _pair(70, 5, O.MATERN52)
    X = torch.rand(batch, mq, 5, generator=torch.Generator().manual_seed(mq),
                   dtype=torch.float64)
    with torch.no_grad():
        post = gp.posterior(X.to(DEV))
        m_r, c_r = orc.posterior(X)
    cov = post.covariance_matrix
    assert (post.mean.squeeze(-1).cpu() - m_r).abs().max() < 1e-10 * m_r.abs().max()
    assert (cov.cpu() - c_r).abs().max() < 1e-10 * c_r.abs().max()
    assert torch.equal(cov, cov.transpose(-1, -2))
    assert torch.equal(post.variance.squeeze(-1), cov.diagonal(dim1=-2, dim2=-1))
