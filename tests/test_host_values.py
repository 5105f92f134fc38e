"""What a model's hyperparameters and outcome statistics may be when they are read to the
host: the scalars are single values (more are refused, as by float()), and only the
posterior needs an outcome transform's statistics."""
import pytest
import torch

import botorch_amd as B
from botorch_amd.fit import ExactMarginalLogLikelihood


def _model(**kw):
    g = torch.Generator().manual_seed(0)
    X = torch.rand(9, 2, generator=g, dtype=torch.float64)
    return B.SingleTaskGP(X, X.sum(-1, keepdim=True), **kw)


@pytest.mark.parametrize("part,name", [("likelihood", "raw_noise"),
                                       ("mean_module", "raw_constant"),
                                       ("covar_module", "raw_outputscale")])
def test_scalars_of_several_values_are_refused(part, name):
    kw = {"covar_module": B.ScaleKernel(B.RBFKernel(ard_num_dims=2))}
    gp = _model(**kw)
    mod = getattr(gp, part)
    setattr(mod, name, torch.nn.Parameter(torch.full((3,), 0.5, dtype=torch.float64)))
    with pytest.raises(RuntimeError, match="3 elements"):
        gp.hyperparameters()
    setattr(mod, name, torch.nn.Parameter(torch.full((1, 1), 0.5, dtype=torch.float64)))
    hp = gp.hyperparameters()  # a single value of any shape is one number
    assert all(isinstance(hp[k], float) for k in ("outputscale", "noise", "constant"))


def test_statistics_of_several_values_are_refused():
    gp = _model()
    gp.outcome_transform.means = torch.zeros(2, 1, dtype=torch.float64)
    with pytest.raises(RuntimeError, match="2 elements"):
        gp.prediction_cache()


class _Shift(torch.nn.Module):
    def forward(self, Y, Yvar=None, X=None):
        return Y - 1.0, Yvar


def test_a_transform_without_statistics_does_not_stop_the_hyperparameters():
    gp = _model(outcome_transform=_Shift())
    hp = gp.hyperparameters()
    assert hp["constant"] == 0.0 and hp["lengthscale"].shape == (2,)
    # the likelihood's only need is the training targets; without a GPU it gets as far as
    # the library
    mll = ExactMarginalLogLikelihood(gp.likelihood, gp)
    if not torch.cuda.is_available():
        with pytest.raises(RuntimeError, match="needs a HIP GPU"):
            mll.loss_and_grads()
    with pytest.raises(AttributeError):
        gp.prediction_cache()
