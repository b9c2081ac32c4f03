"""Rounding of the unwrapping solve, which carries two real lines in one complex transform, against float64 on the same
inputs: at no size and for no right-hand side further off than with one real line per transform."""
import math

import numpy as np
import pytest
import torch
from scipy.fft import dctn, idctn

import ctdm_amd

pytestmark = pytest.mark.gpu

# Mean over 64 maps of |u - u64| / |u64|, in 1e-7, with one real line per transform, measured on these inputs (wrapped and
# sine right-hand side); the solve's may be no larger.
ONE_LINE = {32: (1.566, 1.719), 64: (1.772, 1.970), 128: (1.841, 1.819), 192: (2.294, 2.353), 256: (3.213, 2.918)}


def _maps(N, seed):
    """Four wrapped maps of seven Gaussian bodies with pixel noise."""
    r = np.random.default_rng(1000 * N + seed)
    x = np.arange(N) / N
    p = np.zeros((4, N, N))
    for b in range(4):
        for i in range(7):
            cx, cy = 0.5 + 0.15 * r.uniform(-1, 1, 2)
            s = r.uniform(0.08, 0.12) if i < 2 else r.uniform(0.02, 0.04)
            peak = r.uniform(4, 7) if i < 2 else r.uniform(0.5, 1.5)
            p[b] += peak * np.outer(np.exp(-((x - cy) / s) ** 2 / 2), np.exp(-((x - cx) / s) ** 2 / 2))
    p += 0.025 * r.standard_normal(p.shape)
    return (p - 2 * np.pi * np.round(p / (2 * np.pi))).astype(np.float32)


def _solve64(w, sincos):
    w = w.astype(np.float64)
    rho = np.zeros_like(w)
    for ax in (1, 2):
        d = np.diff(w, axis=ax)
        d = np.sin(d) if sincos else d - 2 * np.pi * np.round(d / (2 * np.pi))
        lo = [slice(None)] * 3
        hi = [slice(None)] * 3
        lo[ax], hi[ax] = slice(None, -1), slice(1, None)
        rho[tuple(lo)] += d
        rho[tuple(hi)] -= d
    e = np.sin(np.pi * np.arange(w.shape[-1]) / (2 * w.shape[-1])) ** 2
    lam = -4 * (e[:, None] + e)
    lam[0, 0] = math.inf
    return idctn(dctn(rho, axes=(1, 2), norm="ortho") / lam, axes=(1, 2), norm="ortho")


@pytest.mark.parametrize("N", sorted(ONE_LINE))
@pytest.mark.parametrize("sincos", [False, True])
def test_error_is_that_of_one_line_per_transform(ctx, N, sincos):
    off = []
    for seed in range(16):
        w = _maps(N, seed)
        u = ctx.unwrap_dct(torch.from_numpy(w).cuda(), ctdm_amd.UNWRAP_SINCOS if sincos else 0).cpu().numpy()
        e = _solve64(w, sincos)
        off += list(np.linalg.norm(u - e, axis=(1, 2)) / np.linalg.norm(e, axis=(1, 2)))
    print(f"{N} sincos {sincos}: {np.mean(off) * 1e7:.3f}e-7")
    assert np.mean(off) <= ONE_LINE[N][sincos] * 1e-7
