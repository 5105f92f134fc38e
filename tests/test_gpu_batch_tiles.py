"""The batched step on both sides of the rule that picks its forward tiles (128 x 128
from 1.75 per CU, 128 x 64 below; 448 tiles on 256 CUs), with models of uneven size:
each model's outputs equal its one-model step's bit for bit."""
import pytest
import torch

import botorch_amd as B

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _acq(n, d, seed):
    g = torch.Generator().manual_seed(seed)
    X = torch.rand(n, d, generator=g, dtype=torch.float64)
    Y = torch.sin(3 * X).sum(-1, keepdim=True)
    Y = Y + 0.01 * torch.randn(n, 1, generator=g, dtype=torch.float64)
    gp = B.SingleTaskGP(X.to(DEV), Y.to(DEV))
    return B.qLogNoisyExpectedImprovement(
        gp, X[:4].to(DEV), sampler=B.SobolQMCNormalSampler(torch.Size([128]), seed=0),
        prune_baseline=False, precision="mixed")


# 1024 points: 8 column tiles; b q = 512: 4 row tiles.  300 points, 130 rows: 3 x 2
@pytest.mark.parametrize("copies,b,q,wide", [(13, 256, 2, False), (14, 256, 2, True),
                                             (19, 130, 1, False), (40, 130, 1, True)])
def test_batch_tiles_equal_one_model_steps(copies, b, q, wide):
    print(f"[case] copies={copies} b={b} q={q} wide={wide}", flush=True)
    base = [_acq(1000, 6, 1), _acq(300, 9, 2)]
    acqs = [base[0]] * copies + [base[1]]
    step = B.BatchedQLogNEI(acqs, b, q)
    tiles = (b * q + 127) // 128 * (8 * copies + 3)
    assert (step.plan.fwd_workers > step.plan.fwd_tiles) == wide == (4 * tiles >= 7 * 256)
    assert step.plan.fwd_tiles == tiles * (1 if wide else 2)
    Xs = [torch.rand(b, q, a.X_baseline.shape[-1], dtype=torch.float64,
                     generator=torch.Generator().manual_seed(i)).to(DEV)
          for i, a in enumerate(acqs)]
    values, grads = step.value_and_grad(Xs)
    for i in (0, copies // 2, copies):
        v, g = acqs[i].value_and_grad(Xs[i])
        assert torch.equal(values[i], v) and torch.equal(grads[i], g)
