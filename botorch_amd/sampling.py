"""Sobol-QMC normal base samples (sampling/normal.py:173-213, sampling/qmc.py:59-97,
utils/sampling.py:51-143).

Base samples come from ``torch.quasirandom.SobolEngine`` - the same engine the
reference uses - followed by the inverse-normal transform with the eps clamp of
sampling/qmc.py:80-83, so they are bit-identical to the reference's for the
same seed; large seeded draws for a GPU (pruning's) come from the same points
formed there (bta_sobol_normal), equal up to the rounding of the transform.
They are generated once per shape (as in the reference); the per-step sampling
(mean + L z) runs in libbotorch_amd.
"""
from __future__ import annotations

import math

import torch
from torch import Tensor
from torch.quasirandom import SobolEngine

from . import _lib
from .exceptions import UnsupportedError


# Draws of at least this many values are formed on the GPU (2048 x 400: 7.4 ms by the
# engine on 16 cores, most of it serial, against 0.7 ms); the smaller ones of an
# acquisition function's base samples (512 x 12: 0.2 ms) keep the engine's bits.
DEVICE_DRAW = 1 << 16
DEVICE_POINTS = 65535 * 64  # of one bta_sobol_normal call


def _scramble_bits(d: int, seed: int) -> Tensor:
    """Host words, also under a default device: the direction numbers (d x 30), the
    scrambling rows (d x 30) and the shifts (d) of bta_sobol_normal."""
    bits = torch.empty(2 * d * 30 + d, dtype=torch.int32, device="cpu")
    cols, rows, shift = bits.split([d * 30, d * 30, d])
    cols.copy_(SobolEngine(dimension=d, scramble=False).sobolstate.reshape(-1))
    _lib.check(_lib.load().bta_sobol_scramble(seed, d, rows.data_ptr(), shift.data_ptr()),
               "sobol_scramble")
    return bits


def _device_normal_samples(d: int, n: int, device, seed: int) -> Tensor:
    L = _lib.lib()
    host = _scramble_bits(d, seed)
    out = torch.empty(n, d, dtype=torch.float64, device=device)
    with torch.cuda.device(out.device):
        bits = host.to(out.device)
        base = bits.data_ptr()
        _lib.check(L.bta_sobol_normal(base, base + 4 * d * 30, base + 8 * d * 30, d, n,
                                      _lib.ptr(out), _lib.stream()), "sobol_normal")
        if torch.get_default_dtype() != torch.float32:
            # the engine keeps its first point (the shift) in the default dtype; the
            # kernel's is the single-precision one
            out[0] = _normal_quantile((host[-d:].to(torch.int64) / 2**30).to(torch.float64)).to(
                out.device)
    return out


def _normal_quantile(u: Tensor) -> Tensor:
    """The inverse-normal transform with the eps clamp of sampling/qmc.py:80-83."""
    v = 0.5 + (1 - torch.finfo(u.dtype).eps) * (u - 0.5)
    return torch.erfinv(2 * v - 1) * math.sqrt(2)


def draw_sobol_normal_samples(d: int, n: int, device=None, dtype=torch.float64,
                              seed: int | None = None) -> Tensor:
    """n x d quasi-normal samples (utils/sampling.py:114-143, qmc.py:80-83)."""
    if (device is not None and torch.device(device).type == "cuda" and dtype == torch.float64
            and type(seed) is int and 0 <= seed < 2**32  # (the engine refuses other types)
            and d * n >= DEVICE_DRAW and n <= DEVICE_POINTS):
        return _device_normal_samples(d, n, device, seed)
    eng = SobolEngine(dimension=d, scramble=True, seed=seed)
    return _normal_quantile(eng.draw(n, dtype=dtype)).to(device=device)


def draw_sobol_samples(bounds: Tensor, n: int, q: int, batch_shape=None,
                       seed: int | None = None) -> Tensor:
    """n x q x d scaled Sobol points in the box ``bounds`` (utils/sampling.py:51-99)."""
    batch_shape = batch_shape or torch.Size()
    batch_size = int(torch.Size(batch_shape).numel())
    d = bounds.shape[-1]
    eng = SobolEngine(q * d, scramble=True, seed=seed)
    raw = eng.draw(batch_size * n, dtype=bounds.dtype)
    raw = raw.view(*batch_shape, n, q, d).to(device=bounds.device)
    if batch_shape != torch.Size():
        raw = raw.permute(-3, *range(len(batch_shape)), -2, -1)
    lo, hi = bounds[0], bounds[1]
    return lo + (hi - lo) * raw


class SobolQMCNormalSampler(torch.nn.Module):
    """Sampler with t-batch-collapsed Sobol base samples (sampling/base.py:32-150)."""

    def __init__(self, sample_shape: torch.Size, seed: int | None = None):
        super().__init__()
        if not isinstance(sample_shape, torch.Size):
            raise UnsupportedError("sample_shape must be a torch.Size")
        self.sample_shape = sample_shape
        self.seed = seed if seed is not None else int(torch.randint(0, 1000000, (1,)).item())
        self.register_buffer("base_samples", None)

    def _get_collapsed_shape(self, posterior) -> torch.Size:
        bss = posterior.base_sample_shape
        start, end = posterior.batch_range
        end = len(bss) + end if end < 0 else end
        return self.sample_shape + torch.Size(
            [1 if start <= i < end else s for i, s in enumerate(bss)])

    def _construct_base_samples(self, posterior) -> None:
        target = self._get_collapsed_shape(posterior)
        if self.base_samples is None or self.base_samples.shape != target:
            out_dim = target[len(self.sample_shape):].numel()
            if out_dim > SobolEngine.MAXDIM:
                raise UnsupportedError(
                    f"SobolQMCSampler only supports dimensions q * o <= {SobolEngine.MAXDIM}")
            bs = draw_sobol_normal_samples(out_dim, self.sample_shape.numel(),
                                           device=posterior.device, dtype=posterior.dtype,
                                           seed=self.seed)
            self.base_samples = bs.view(target)

    def forward(self, posterior) -> Tensor:
        self._construct_base_samples(posterior)
        return posterior.rsample_from_base_samples(
            self.sample_shape,
            self.base_samples.expand(self.sample_shape + posterior.base_sample_shape))


def get_sampler(posterior, sample_shape: torch.Size, seed: int | None = None):
    return SobolQMCNormalSampler(sample_shape=sample_shape, seed=seed)
