"""The positivity loop's two passes over the volume, each holding half of the y transform, against the loop
in double precision (numpy): every volume side and tile size, lists of every length, and a volume that starts 8
bytes past a 16-byte boundary.

Tolerance: an FP32 transform of 3 log2(V) <= 24 stages carries a relative rounding of about 6e-8 sqrt(24) = 3e-7
of the rms, 5 sigma over the volume 1.5e-6; there are two per iteration. With |f| / k^2 <= 0.05 and
n = n_m sqrt(1 - f / k^2) that is 1.34 * 0.5 * 0.05 * 3e-6 = 1e-7 in n, per iteration, beside the 1.2e-7 resolution of n near
1.34 itself. Three iterations: 5e-7; the bar is twice that."""
import numpy as np
import pytest
import torch

import ctdm_amd

pytestmark = pytest.mark.gpu
LAM, NM = 532e-9, 1.337
TOL = 1e-6


@pytest.fixture(scope="module")
def ctx():
    c = ctdm_amd.Context()
    yield c
    c.close()


def est_n(f, k2):
    n = NM * np.sqrt(1 - f / k2 + 0j)
    return np.maximum(n.real, NM) + 1j * np.maximum(n.imag, 0)


def loop(f, Fm, mask, iters, k2):
    n = est_n(f, k2)
    for _ in range(iters):
        F = np.fft.fftn(-k2 * ((n / NM) ** 2 - 1))
        F[mask] = Fm[mask]
        n = est_n(np.fft.ifftn(F), k2)
    return n


def case(V, seed, fill):
    rng = np.random.default_rng(seed)
    k2 = (2 * np.pi * NM / LAM) ** 2
    f = 0.02 * k2 * np.clip(rng.standard_normal((V, V, V)) + 1j * rng.standard_normal((V, V, V)), -2.5, 2.5)
    f = f.astype(np.complex64)
    F = np.fft.fftn(f.astype(np.complex128))
    F *= rng.uniform(0.9, 1.1, (V, V, V))
    # `fill` of each z pencil is measured: none (0), a length that differs from pencil to pencil, or all (1)
    part = rng.uniform(0, 2 * fill, (V, V)) if 0 < fill < 1 else np.full((V, V), fill)
    mask = rng.uniform(size=(V, V, V)) < part[None]
    return f, np.where(mask, F, 0).astype(np.complex64), mask, k2


def cuda(a, off=0):
    """`a` on the GPU, `off` elements into its allocation."""
    buf = torch.empty(a.size + off, dtype=torch.from_numpy(a).dtype, device="cuda")
    t = buf[off:].view(a.shape)
    t.copy_(torch.from_numpy(a))
    return t


@pytest.mark.parametrize("V,iters,fill", [(32, 1, 0.5), (32, 3, 0.2), (64, 3, 0.3), (64, 1, 0.0), (64, 2, 1.0), (128, 2, 0.2),
                                          (192, 1, 0.4), (256, 2, 0.15)])
def test_two_pass_loop(ctx, V, iters, fill):
    f, Fm, mask, k2 = case(V, V + iters, fill)
    want = loop(f.astype(np.complex128), Fm.astype(np.complex128), mask, iters, k2)
    o = ctdm_amd.Optics(LAM, NM, 0.1e-6)
    Fd, hd = cuda(Fm), cuda(mask.astype(np.float32))
    saved = ctx.get_tuning(V)
    first = None
    try:
        for px, pz, off in ((16, 16, 0), (8, 16, 1), (16, 8, 0), (8, 8, 1)):
            ctx.set_tuning(V, (px, 16, pz, 8), (px // 16, 0), 0)
            n = ctx.positivity(cuda(f, off), Fd, hd, iters, o, ctdm_amd.POS_NO_SHIFT)
            if first is None:
                first = n
                e = float(np.abs(n.cpu().numpy() - want).max())
                print(f"V={V}, {iters} iterations, fill {fill}: max|dn| {e:.1e}")
                assert e <= TOL
            assert torch.equal(n, first), (px, pz, off)  # tile sizes and directions change no value
    finally:
        ctx.set_tuning(V, saved["pencils"], saved["sweep"], saved["yplan"])


def test_projection_over_its_branches(ctx):
    """One iteration with nothing measured gives est_n of the projection of f: 1 - f / k^2 over [-2, 3] x [-2, 2], with
    zeros and the branch point, and a NaN voxel, which projects to 0. The volume's rms is 2 k^2, so its two
    transforms leave 1.34 * 0.5 * 2 * 5 * 3e-7 * sqrt(2) = 3e-6 in n (|sqrt| >= 1 after the clamps); the bar is twice that."""
    V = 64
    k2 = (2 * np.pi * NM / LAM) ** 2
    rng = np.random.default_rng(3)
    c, d = rng.uniform(-2, 3, (V, V, V)), rng.uniform(-2, 2, (V, V, V))
    f = (k2 * ((1 - c) - 1j * d)).astype(np.complex64)
    f[0, 0, :3] = 0, np.float32(k2), np.float32(2 * k2)
    f[1, 0, 0] = complex(0.5 * k2, 0)
    g = f.copy()
    g[2, 0, 0] = complex(np.nan, np.nan)
    f[2, 0, 0] = 0
    z = f.astype(np.complex128)
    z.imag[z.imag == 0] = 0.0
    want = est_n(z, k2)
    none = torch.zeros((V, V, V), dtype=torch.float32, device="cuda")
    o = ctdm_amd.Optics(LAM, NM, 0.1e-6)
    for src in (f, g):
        n = ctx.positivity(cuda(src), torch.zeros_like(cuda(f)), none, 1, o, ctdm_amd.POS_NO_SHIFT).cpu().numpy()
        e = np.abs(n - want)
        e[0, 0, 1:3] = 0  # at the cut itself the sign of a zero decides
        print(f"max|dn| {e.max():.1e}")
        assert e.max() <= 6e-6


@pytest.mark.parametrize("V,fill", [(32, 0.0), (32, 1.0), (64, 0.1), (192, 0.3)])
def test_measured_list_by_value(ctx, V, fill):
    """The list of CTDM_DC_REFCOMPAT: voxels whose real and imaginary parts both differ from zero, some with one zero part;
    one iteration against the loop in double precision (tolerance as above)."""
    f, Fm, mask, k2 = case(V, 7 + V, fill)
    Fm[:, :, ::7] = 1j * Fm[:, :, ::7].imag
    Fm[:, ::5] = Fm[:, ::5].real
    mask = (Fm.real != 0) & (Fm.imag != 0)
    want = loop(f.astype(np.complex128), Fm.astype(np.complex128), mask, 1, k2)
    n = ctx.positivity(cuda(f), cuda(Fm), None, 1, ctdm_amd.Optics(LAM, NM, 0.1e-6),
                       ctdm_amd.POS_NO_SHIFT | ctdm_amd.DC_REFCOMPAT)
    assert float(np.abs(n.cpu().numpy() - want).max()) <= TOL
