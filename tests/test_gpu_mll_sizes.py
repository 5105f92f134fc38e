"""The MLL value and gradient over the sizes where its path changes (32 x 32 trace
tiles and 64-point padding up to trs_max_n, 128 x 64 tiles above; 8, 16 and 32
coordinate slots; 4- and 16-row covariance blocks) against the FP64 oracle's closed
form.

Tolerance: both sides are FP64 and differ by rounding amplified by cond(K) <= (n s +
noise) / noise ~ 3e5: 1e-9 of the value and of the largest gradient entry."""
import ctypes
import math

import pytest
import torch

from botorch_amd import _lib
from oracle import gp_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,d,kind", [
    (2, 1, O.RBF), (31, 8, O.MATERN52), (32, 9, O.RBF), (33, 3, O.MATERN52), (64, 16, O.RBF),
    (65, 17, O.MATERN52), (129, 32, O.RBF), (1024, 8, O.MATERN52), (1025, 5, O.RBF),
    (2049, 17, O.MATERN52), (3072, 16, O.RBF), (3073, 16, O.MATERN52)])
def test_mll_sizes_match_oracle(n, d, kind):
    print(f"[case] n={n} d={d} kind={kind}", flush=True)
    g = torch.Generator().manual_seed(n + d)
    X = torch.rand(n, d, generator=g, dtype=torch.float64)
    y = torch.sin(3 * X).sum(-1) + 0.05 * torch.randn(n, generator=g, dtype=torch.float64)
    y = (y - y.mean()) / y.std()
    ls = 0.3 + torch.rand(d, generator=g, dtype=torch.float64)
    s, noise, c = 1.3, 1e-2, 0.2
    L = _lib.lib()
    need = L.bta_mll_workspace_size(n, d)
    ws = _lib.workspace(need, "cuda")
    out = (ctypes.c_double * (4 + d))()
    Xd, yd = X.cuda(), y.cuda()
    for _ in range(2):  # the second call finds the first one's workspace
        _lib.check(L.bta_mll_value_grad(kind, _lib.ptr(Xd), _lib.ptr(yd), n, d,
                                        (ctypes.c_double * d)(*ls.tolist()), s, noise, c, 6, out,
                                        _lib.ptr(ws), ws.numel(), _lib.stream()), "mll")
    K = O.covar_direct(kind, X, X, ls, s) if n <= 1100 else O.covar(kind, X, X, ls, s)
    Lc = torch.linalg.cholesky(K + noise * torch.eye(n, dtype=torch.float64))
    r = (y - c).unsqueeze(-1)
    a = torch.cholesky_solve(r, Lc)
    ll = -0.5 * ((r * a).sum() + 2 * torch.log(torch.diagonal(Lc)).sum()
                 + n * math.log(2 * math.pi))
    W = a @ a.t() - torch.cholesky_inverse(Lc)
    g_ls = []
    for j in range(d):
        sq = (X[:, None, j] - X[None, :, j]) ** 2
        g_ls.append(sq)
    r2 = sum(q / l**2 for q, l in zip(g_ls, ls))
    if kind == O.MATERN52:
        rr = math.sqrt(5) * r2.sqrt()
        h = s * 5.0 / 3.0 * (1 + rr) * torch.exp(-rr)
    else:
        h = s * torch.exp(-0.5 * r2)
    want = [0.5 * (W * K).sum() / s, 0.5 * torch.diagonal(W).sum(), a.sum()]
    want += [0.5 * (W * h * q).sum() / l**3 for q, l in zip(g_ls, ls)]
    want, got = torch.stack(want), torch.tensor(list(out)[1:], dtype=torch.float64)
    assert abs(out[0] - ll.item()) < 1e-9 * max(abs(ll.item()), 1.0)
    assert (got - want).abs().max() < 1e-9 * want.abs().max()
