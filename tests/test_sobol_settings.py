"""Base samples formed on the GPU under other settings of the process: they follow
torch's SobolEngine for every default dtype and default device, and take the seeds that
it takes.

Tolerance of the draw: the points are equal and the two inverse error functions are each
within a few ulp of |z| <= 6.3: 4e-15 absolute."""
import math

import numpy as np
import pytest
import torch
from torch.quasirandom import SobolEngine

from botorch_amd import sampling


@pytest.fixture
def default_dtype():
    before = torch.get_default_dtype()
    yield torch.set_default_dtype
    torch.set_default_dtype(before)


def _engine(d, n, seed):
    u = SobolEngine(dimension=d, scramble=True, seed=seed).draw(n, dtype=torch.float64)
    v = 0.5 + (1 - torch.finfo(torch.float64).eps) * (u - 0.5)
    return torch.erfinv(2 * v - 1) * math.sqrt(2)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.bfloat16])
@pytest.mark.parametrize("d,n", [(700, 100), (SobolEngine.MAXDIM, 4)])
def test_device_draw_follows_the_default_dtype(default_dtype, dtype, d, n):
    print(f"[case] {dtype} d={d} n={n}", flush=True)
    default_dtype(dtype)
    z = sampling.draw_sobol_normal_samples(d, n, device="cuda", seed=7)
    ref = _engine(d, n, 7)
    assert d * n >= sampling.DEVICE_DRAW and z.dtype == torch.float64
    assert torch.isfinite(ref).all()
    assert (z.cpu() - ref).abs().max() < 4e-15


def test_scrambling_bits_are_host_words_under_any_default_device():
    with torch.device("meta"):  # a GPU default would hand a device pointer to host code
        bits = sampling._scramble_bits(3, 11)
    assert bits.device.type == "cpu" and bits.dtype == torch.int32
    shift = SobolEngine(dimension=3, scramble=True, seed=11).shift
    assert torch.equal(bits[-3:].to(torch.int64), shift)


@pytest.mark.gpu
def test_device_draw_under_a_default_device():
    z = sampling.draw_sobol_normal_samples(512, 128, device="cuda", seed=3)
    with torch.device("cuda"):
        again = sampling.draw_sobol_normal_samples(512, 128, device="cuda", seed=3)
    assert torch.equal(z, again)


@pytest.mark.parametrize("seed", [np.int64(3), 3.0, True, np.array(3), torch.tensor(3)])
def test_seeds_the_engine_refuses_are_refused(seed):
    for device in ("cpu", "cuda"):
        with pytest.raises((TypeError, RuntimeError), match="integer|manual_seed"):
            sampling.draw_sobol_normal_samples(512, 128, device=device, seed=seed)
