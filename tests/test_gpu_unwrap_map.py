"""The whole solve of a small map in one workgroup (32^2 and 64^2): both right-hand sides, both eigenvalue tables and the
congruence step against float64, inputs and outputs at any float of a buffer, and maps of a large call equal to the same
maps alone."""
import math

import numpy as np
import pytest
import torch

import ctdm_amd

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


def solution(w, flags):
    N = w.shape[-1]
    n = np.arange(N)
    D = np.cos(np.pi * (2 * n[None] + 1) * n[:, None] / (2 * N)) * math.sqrt(2 / N)
    D[0] = math.sqrt(1 / N)
    lam = (2 * np.cos(4 * np.pi * n / (4 * N - 1))[:, None] + 2 * np.cos(4 * np.pi * n / (4 * N - 1))[None] - 4
           if flags & ctdm_amd.UNWRAP_REFCOMPAT_EIG else
           -4 * (np.sin(np.pi * n / (2 * N)) ** 2 + (np.sin(np.pi * n / (2 * N)) ** 2)[:, None]))
    lam[0, 0] = 1
    step = np.sin if flags & ctdm_amd.UNWRAP_SINCOS else lambda d: (d + np.pi) % (2 * np.pi) - np.pi
    rho = np.zeros_like(w)
    for ax in (-1, -2):
        d = step(np.diff(w, axis=ax))
        lo, hi = [slice(None)] * 3, [slice(None)] * 3
        lo[ax], hi[ax] = slice(None, -1), slice(1, None)
        rho[tuple(lo)] += d
        rho[tuple(hi)] -= d
    X = D @ rho @ D.T / lam
    X[..., 0, 0] = 0
    return D.T @ X @ D


def maps(N, batch, seed):
    rng = np.random.default_rng(seed)
    y, x = np.mgrid[0:N, 0:N] / N
    c = rng.uniform(0.3, 0.7, (batch, 2, 1, 1))
    phi = 7 * np.exp(-((x - c[:, 0]) ** 2 + (y - c[:, 1]) ** 2) / 0.05) + 0.2 * rng.standard_normal((batch, N, N))
    return np.angle(np.exp(1j * phi)).astype(np.float32)


@pytest.mark.parametrize("N", [32, 64])
@pytest.mark.parametrize("flags", [0, ctdm_amd.UNWRAP_SINCOS, ctdm_amd.UNWRAP_REFCOMPAT_EIG,
                                   ctdm_amd.UNWRAP_CONGRUENT, ctdm_amd.UNWRAP_SINCOS | ctdm_amd.UNWRAP_CONGRUENT])
def test_map_solve(ctx, N, flags):
    w = maps(N, 5, N + flags)
    v = solution(w.astype(np.float64), flags)
    buf = torch.zeros(2, w.size + 3, device="cuda")
    ref = None
    for off in (0, 1, 3):
        src, dst = buf[0, off:off + w.size], buf[1, 3 - off:3 - off + w.size]
        src.copy_(torch.from_numpy(w.reshape(-1)))
        ctx._call("ctdm_unwrap_dct", src.data_ptr(), dst.data_ptr(), 5, N, flags)
        got = dst.cpu().numpy().reshape(w.shape)
        ref = got if ref is None else ref
        assert np.array_equal(got, ref), off
    # four transforms of log2 N stages, each rounding to eps of the solution's largest values; a difference within one eps
    # of +-pi may wrap the other way, which these maps' noise makes a matter of luck below 1e-5 per map
    tol = 16 * math.log2(N) * EPS * np.abs(v).max()
    if flags & ctdm_amd.UNWRAP_CONGRUENT:
        k = (ref - w.astype(np.float64)) / (2 * np.pi)
        assert np.abs(k - np.round(k)).max() <= 4 * EPS * np.abs(ref).max() / (2 * np.pi) + 1e-6
        assert np.abs(ref - v).max() <= np.pi + tol + 1e-5
    else:
        err = np.abs(ref - v).max()
        print(f"N={N} flags {flags}: max err {err:.1e}, bar {tol:.1e}")
        assert err <= tol
    many = torch.from_numpy(np.concatenate([maps(N, 300, 9), w])).cuda()
    assert np.array_equal(ctx.unwrap_dct(many, flags)[300:].cpu().numpy(), ref)
