"""The qLogNEI value+grad step at the edges of its elementwise stages (row and column
tiles of 64, restarts that straddle a wave's 16 rows, 16 columns of [alpha | A] in LDS,
baselines of 15..70 points, every coordinate block) against the FP64 oracle.

Tolerance: the samples carry about cond(K) eps ~ 1e4 x 2e-16 x 10; the log of the
smoothed improvement divides that by tau_relu = 1e-6: 2e-5 of the largest entry covers
both the value and the gradient."""
import pytest
import torch

import botorch_amd as B
from oracle import gp_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("n,d,q,n_b,b,S,kind", [
    (40, 1, 1, 1, 1, 64, O.RBF), (63, 4, 7, 15, 9, 96, O.MATERN52), (64, 5, 5, 16, 13, 128, O.RBF),
    (65, 8, 6, 17, 11, 130, O.MATERN52), (200, 13, 3, 40, 43, 256, O.MATERN52),
    (193, 32, 8, 70, 9, 256, O.RBF), (130, 17, 2, 3, 65, 600, O.MATERN52),
    (70, 2, 4, 7, 16, 256, O.RBF)])
def test_step_edges_match_oracle(n, d, q, n_b, b, S, kind):
    print(f"[case] n={n} d={d} q={q} n_b={n_b} b={b} S={S} kind={kind}", flush=True)
    g = torch.Generator().manual_seed(n + 31 * q)
    X = torch.rand(n, d, generator=g, dtype=torch.float64)
    Y = torch.sin(3 * X).sum(-1, keepdim=True)
    Y = Y + 0.1 * torch.randn(n, 1, generator=g, dtype=torch.float64)
    ls = (0.3 + 0.7 * torch.rand(d, generator=g, dtype=torch.float64)) * max(1.0, (d / 6) ** 0.5)
    base = (B.MaternKernel if kind == O.MATERN52 else B.RBFKernel)(ard_num_dims=d)
    base.lengthscale = ls
    lik = B.GaussianLikelihood()
    lik.noise = 1e-2
    covar = B.ScaleKernel(base)
    covar.outputscale = 1.0
    gp = B.SingleTaskGP(X.to(DEV), Y.to(DEV), likelihood=lik, covar_module=covar)
    orc = O.OracleGP(X, Y, kind, ls, 1.0, 1e-2)
    acq = B.qLogNoisyExpectedImprovement(gp, X[:n_b].to(DEV),
                                         sampler=B.SobolQMCNormalSampler(torch.Size([S]), seed=0),
                                         prune_baseline=False)
    ref = O.OracleQLogNEI(orc, X[:n_b], num_samples=S, seed=0)
    Xq = torch.rand(b, q, d, generator=g, dtype=torch.float64)
    v_ref, g_ref = ref.value_and_grad(Xq)
    v, gr = acq.value_and_grad(Xq.to(DEV))
    assert (v.cpu() - v_ref).abs().max() <= 2e-5 * v_ref.abs().max()
    assert (gr.cpu() - g_ref).abs().max() <= 2e-5 * g_ref.abs().max()
    with torch.no_grad():
        assert torch.equal(acq(Xq.to(DEV)), v)  # value alone


@pytest.mark.parametrize("n,q,b,S", [(64, 1, 32, 512), (130, 3, 11, 64), (1011, 3, 200, 256),
                                     (200, 8, 40, 128), (64, 2, 3000, 64)])
def test_fused_fp64_adjoint_matches_sequential(n, q, b, S, monkeypatch):
    # the FP64 MC stage and U = V L^-1 in one launch against one after the other: the
    # same arithmetic but for the number of partial sums per entry of U (4 or 8), so
    # a few ulp of the largest gradient entry: 1e-12
    print(f"[case] n={n} q={q} b={b} S={S}", flush=True)
    g = torch.Generator().manual_seed(n)
    X = torch.rand(n, 6, generator=g, dtype=torch.float64)
    Y = torch.sin(3 * X).sum(-1, keepdim=True)
    gp = B.SingleTaskGP(X.to(DEV), Y.to(DEV))
    acq = B.qLogNoisyExpectedImprovement(gp, X[:9].to(DEV),
                                         sampler=B.SobolQMCNormalSampler(torch.Size([S]), seed=0),
                                         prune_baseline=False)
    Xq = torch.rand(b, q, 6, generator=g, dtype=torch.float64).to(DEV)
    v, gr = acq.value_and_grad(Xq)
    monkeypatch.setenv("BTA_SEQUENTIAL_ADJOINT", "1")
    v2, gr2 = acq.value_and_grad(Xq)
    assert torch.equal(v, v2)
    assert (gr - gr2).abs().max() <= 1e-12 * gr2.abs().max()
