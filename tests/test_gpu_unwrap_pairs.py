"""Unwrapping kernels that transform two real lines as one complex line, and the adjoint that leaves out the
Laplacian of the Poisson solution: every size, odd batches, inputs beyond one period, buffers at odd addresses
and in-place gradients, against float64 references."""
import math

import numpy as np
import pytest
import torch

import ctdm_amd

pytestmark = pytest.mark.gpu
SIZES = [32, 64, 128, 192, 256]
EPS = 2.0 ** -24


def _poisson(rho, refeig=False):
    N = rho.shape[-1]
    n = np.arange(N)
    D = np.cos(np.pi * (2 * n[None] + 1) * n[:, None] / (2 * N)) * math.sqrt(2 / N)
    D[0] = math.sqrt(1 / N)
    lam = (2 * np.cos(4 * np.pi * n / (4 * N - 1))[:, None] + 2 * np.cos(4 * np.pi * n / (4 * N - 1))[None] - 4
           if refeig else -4 * (np.sin(np.pi * n / (2 * N)) ** 2 + (np.sin(np.pi * n / (2 * N)) ** 2)[:, None]))
    lam[0, 0] = 1
    X = D @ rho @ D.T / lam
    X[..., 0, 0] = 0
    return D.T @ X @ D


def _stencil(v, w=None):
    out = np.zeros_like(v)
    for ax in (-1, -2):
        d = np.diff(v, axis=ax)
        if w is not None:
            d = d * np.cos(np.diff(w, axis=ax))
        lo = [slice(None)] * v.ndim
        hi = [slice(None)] * v.ndim
        lo[ax], hi[ax] = slice(None, -1), slice(1, None)
        out[tuple(lo)] += d
        out[tuple(hi)] -= d
    return out


def _phase(N, batch, seed, amp=3.0, noise=0.05):
    rng = np.random.default_rng(seed)
    y, x = np.mgrid[0:N, 0:N].astype(np.float64)
    c = rng.uniform(0.3 * N, 0.7 * N, (batch, 2, 1, 1))
    phi = amp * np.exp(-((x - c[:, 0]) ** 2 + (y - c[:, 1]) ** 2) / (0.04 * N * N))
    phi = phi + noise * rng.standard_normal((batch, N, N))
    return np.angle(np.exp(1j * phi)).astype(np.float32)


@pytest.mark.parametrize("N", SIZES)
@pytest.mark.parametrize("flags", [0, ctdm_amd.UNWRAP_REFCOMPAT_EIG, ctdm_amd.UNWRAP_SINCOS,
                                   ctdm_amd.UNWRAP_SINCOS | ctdm_amd.UNWRAP_REFCOMPAT_EIG])
def test_adjoint_matches_float64(ctx, N, flags):
    w = _phase(N, 3, N + flags)
    g = np.random.default_rng(N).standard_normal(w.shape).astype(np.float32)
    refeig, sincos = flags & ctdm_amd.UNWRAP_REFCOMPAT_EIG, flags & ctdm_amd.UNWRAP_SINCOS
    v = _poisson(g.astype(np.float64), refeig)
    ref = _stencil(v, w.astype(np.float64) if sincos else None)
    wd, gd = torch.from_numpy(w).cuda(), torch.from_numpy(g).cuda()
    got = ctx.unwrap_dct_adjoint(wd, gd, flags).cpu().numpy()
    # each of the (up to) four transforms rounds to about log2 N eps of its largest values: those of the result
    # itself without SINCOS; the solution's differences (four of them, two roundings each) with it
    tol = 16 * math.log2(N) * EPS * (np.abs(g).max() + (np.abs(v).max() if sincos else 0.0))
    err = np.abs(got - ref).max()
    print(f"N={N} flags {flags}: max err {err:.2e}, bar {tol:.2e}")
    assert err <= tol
    ctdm_amd.lib()
    ctx._call("ctdm_unwrap_dct_adjoint", wd.data_ptr(), gd.data_ptr(), gd.data_ptr(), 3, N, flags)  # in place
    assert np.array_equal(gd.cpu().numpy(), got)


@pytest.mark.parametrize("N", SIZES)
@pytest.mark.parametrize("flags", [0, ctdm_amd.UNWRAP_SINCOS | ctdm_amd.UNWRAP_CONGRUENT])
def test_odd_addresses_give_the_same_bits(ctx, N, flags):
    """Maps and results one float past a 16-byte boundary: the four-pixel loads and stores are not aligned."""
    w = torch.from_numpy(_phase(N, 3, 7 * N)).cuda()
    want = ctx.unwrap_dct(w, flags)
    n = w.numel()
    src, dst = torch.zeros(n + 4, device="cuda"), torch.full((n + 4,), -7.0, device="cuda")
    src[1:n + 1] = w.reshape(-1)
    ctx._call("ctdm_unwrap_dct", src.data_ptr() + 4, dst.data_ptr() + 4, 3, N, flags)
    assert torch.equal(dst[1:n + 1].view(3, N, N), want)
    assert dst[0] == -7.0 and (dst[n + 1:] == -7.0).all()
    ga = ctx.unwrap_dct_adjoint(w, want, flags & ctdm_amd.UNWRAP_SINCOS)
    src2 = torch.zeros(n + 4, device="cuda")
    src2[1:n + 1] = want.reshape(-1)
    ctx._call("ctdm_unwrap_dct_adjoint", src.data_ptr() + 4, src2.data_ptr() + 4, dst.data_ptr() + 4, 3, N,
              flags & ctdm_amd.UNWRAP_SINCOS)
    assert torch.equal(dst[1:n + 1].view(3, N, N), ga)


@pytest.mark.parametrize("N", [32, 192, 256])
def test_differences_beyond_the_wrapped_range(ctx, orc, N):
    """Maps of +-15 rad: differences up to 30 rad take the wrap's general formula beside the short one."""
    w = np.random.default_rng(N).uniform(-15, 15, (2, N, N)).astype(np.float32)
    got = ctx.unwrap_dct(torch.from_numpy(w).cuda()).cpu().numpy()
    ref = orc.unwrap_dct(w.astype(np.float64))
    # a difference within a few ulp of an odd multiple of pi may wrap the other way than in float64 (about
    # 4 N^2 differences, 2e-6 of a period each): at most a handful of unit dipoles of 2 pi, which the solution
    # spreads; everything else is rounding
    err = np.abs(got - ref)
    assert np.median(err) <= 64 * EPS * np.abs(ref).max() and err.max() <= 2 * math.pi
