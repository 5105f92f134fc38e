"""The native Sobol base samples: the scrambling bits and direction numbers against
torch's SobolEngine (bit for bit, on the CPU) and the device draw against the
engine's points through the same transform.

Tolerance of the draw: the points are equal, the two inverse error functions are
each within a few ulp and |z| <= 6.3: 4e-15 absolute."""
import math

import numpy as np
import pytest
import torch
from torch.quasirandom import SobolEngine

from botorch_amd import _lib, sampling


@pytest.mark.parametrize("d,seed", [(1, 0), (7, 1234), (65, 2**32 - 1)])
def test_scrambled_state_equals_the_engines(d, seed):
    rows, shift = np.zeros((d, 30), np.uint32), np.zeros(d, np.uint32)
    _lib.check(_lib.load().bta_sobol_scramble(seed, d, rows.ctypes.data, shift.ctypes.data))
    eng = SobolEngine(dimension=d, scramble=True, seed=seed)
    cols = SobolEngine(dimension=d, scramble=False).sobolstate.numpy().astype(np.uint32)
    v = rows[:, None, :] & cols[:, :, None]  # parity of each row with each column
    for s in (16, 8, 4, 2, 1):
        v = v ^ (v >> np.uint32(s))
    state = ((v & 1).astype(np.int64) << (29 - np.arange(30))).sum(-1)
    assert np.array_equal(state, eng.sobolstate.numpy())
    # point 0 is the shift (in single precision), point i follows by column ctz(i)
    pts = (eng.draw(9, dtype=torch.float64).numpy() * 2**30).astype(np.int64)
    x = shift.astype(np.int64)
    for i in range(9):
        want = x.astype(np.float32).astype(np.int64) if i == 0 else x
        assert np.array_equal(pts[i], want)
        b = ((i + 1) & -(i + 1)).bit_length() - 1
        x = x ^ state[:, b]


@pytest.mark.gpu
@pytest.mark.parametrize("d,n", [(400, 2048), (32, 2048), (65, 1009), (64, 1025), (1, 65536),
                                 (2000, 33)])
def test_device_draw_matches_the_engine(d, n):
    print(f"[case] d={d} n={n}", flush=True)
    z = sampling.draw_sobol_normal_samples(d, n, device="cuda", seed=d + n)
    u = SobolEngine(dimension=d, scramble=True, seed=d + n).draw(n, dtype=torch.float64)
    v = 0.5 + (1 - torch.finfo(torch.float64).eps) * (u - 0.5)
    ref = torch.erfinv(2 * v - 1) * math.sqrt(2)
    assert z.shape == ref.shape and torch.isfinite(z).all()
    assert (z.cpu() - ref).abs().max() < 4e-15
