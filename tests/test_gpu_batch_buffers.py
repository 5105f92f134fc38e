"""The batched step's buffers: what a caller may pass to value_and_grad and what it may
do with the buffers and the results.  Every compared pair runs the same kernels on the
same inputs: equal bit for bit."""
import pytest
import torch

import botorch_amd as B

pytestmark = pytest.mark.gpu
DEV = "cuda"
B_RESTARTS = [3, 5, 2]


def _step():
    acqs = []
    for i, n in enumerate((20, 33, 64)):
        g = torch.Generator().manual_seed(n)
        X = torch.rand(n, 2 + i, generator=g, dtype=torch.float64)
        Y = torch.sin(5 * X).sum(-1, keepdim=True)
        acqs.append(B.qLogNoisyExpectedImprovement(
            B.SingleTaskGP(X.to(DEV), Y.to(DEV)), X[:4].to(DEV), prune_baseline=False,
            precision="mixed", sampler=B.SobolQMCNormalSampler(torch.Size([64]), seed=1)))
    return B.BatchedQLogNEI(acqs, B_RESTARTS, 2)


def _points(step, seed):
    g = torch.Generator().manual_seed(seed)
    return [torch.rand(x.shape, generator=g, dtype=torch.float64).to(DEV) for x in step.X]


def _same(a, b):
    return all(torch.equal(x, y) for p, q in zip(a, b) for x, y in zip(p, q))


def test_inputs_may_be_the_steps_own_buffers():
    step = _step()
    Xs = _points(step, 0)
    want = step.value_and_grad(Xs)
    for buf, X in zip(step.X, Xs):
        buf.copy_(X)
    assert _same(step.value_and_grad(step.X), want)
    assert _same(step.value_and_grad([x[:] for x in step.X]), want)
    # one model's buffer, the others from elsewhere
    assert _same(step.value_and_grad([Xs[0], step.X[1], Xs[2]]), want)


@pytest.mark.parametrize("kind", ["plain", "strided", "float32", "cpu", "expanded"])
@pytest.mark.parametrize("grad", [False, True])
def test_inputs_of_any_type_device_and_layout(kind, grad):
    step = _step()
    Xs = _points(step, 1)
    if kind == "strided":
        given = [x.transpose(0, 1).contiguous().transpose(0, 1) for x in Xs]
    elif kind == "float32":
        given = [x.float() for x in Xs]
        Xs = [x.double() for x in given]
    elif kind == "cpu":
        given = [x.cpu() for x in Xs]
    elif kind == "expanded":
        given = [x[:1] for x in Xs]
        Xs = [x[:1].expand_as(x).contiguous() for x in Xs]
    else:
        given = [x.clone() for x in Xs]
    want = step.value_and_grad(Xs)
    got = step.value_and_grad([x.requires_grad_(grad) for x in given])
    assert _same(got, want)
    assert not any(t.requires_grad for part in got for t in part)


def test_buffers_take_points_that_require_grad():
    step = _step()
    Xs = _points(step, 2)
    want = step.value_and_grad(Xs)
    for buf, X in zip(step.X, Xs):
        buf.copy_(X.clone().requires_grad_(True))
    step.launch()
    assert _same([step.value, step.grad], want)
    assert _same(step.value_and_grad(_points(step, 2)), want)


def test_results_are_independent_of_each_other_and_of_the_buffers():
    """Editing or keeping one model's result touches no other's: own storage, own
    version counter (a graph that saved another result stays valid)."""
    step = _step()
    Xs = _points(step, 3)
    values, grads = step.value_and_grad(Xs)
    parts = values + grads
    assert len({t.untyped_storage().data_ptr() for t in parts + step.value + step.grad}) == 12
    assert all(t.untyped_storage().nbytes() == t.numel() * 8 for t in parts)
    w = torch.ones_like(grads[0], requires_grad=True)
    loss = (w * grads[0]).sum()  # saves grads[0]
    kept = [t.clone() for t in parts]
    for t in values + grads[1:]:
        t.mul_(2.0)
    loss.backward()
    assert torch.equal(w.grad, grads[0])
    again = step.value_and_grad(Xs)
    assert _same(again, [kept[:3], kept[3:]])


def test_a_failed_models_results_come_from_the_joint_posterior():
    step = _step()
    Xs = _points(step, 4)
    want = step.value_and_grad(Xs)
    step.acqfs[1]._keep["Lb"].zero_()
    with pytest.warns(B.BotorchWarning, match="Falling back"):
        v1, g1 = step.acqfs[1].value_and_grad(Xs[1])
    with pytest.warns(B.BotorchWarning, match="Falling back"):
        values, grads = step.value_and_grad(Xs)
    assert torch.equal(values[1], v1) and torch.equal(grads[1], g1)
    assert torch.equal(step.value[1], v1) and torch.equal(step.grad[1], g1)
    for i in (0, 2):
        assert torch.equal(values[i], want[0][i]) and torch.equal(grads[i], want[1][i])
