"""Branch cuts of maps of few columns, which one wavefront draws one residue after the other, against the host
specification: integers and phases follow from the pairing, so every output must be equal bit for bit (tolerance zero)."""
import time

import numpy as np
import pytest
import torch

import ctdm_amd

pytestmark = pytest.mark.gpu


def _equal(ctx, orc, w):
    got = [t.cpu().numpy() for t in ctx.goldstein(torch.from_numpy(w).cuda())]
    for name, g, r in zip(("residues", "cuts", "k2pi", "unwrapped"), got, orc.goldstein(w)):
        assert np.array_equal(g.view(np.uint32) if g.dtype == np.float32 else g,
                              r.view(np.uint32) if r.dtype == np.float32 else r), name
    return got[0]


def _noisy(rng, shape, noise):
    """Wrapped maps of a slope plus uniform noise of +-noise pi."""
    B, H, W = shape
    y, x = np.mgrid[0:H, 0:W]
    p = 0.05 * x + 0.02 * y + rng.uniform(-noise * np.pi, noise * np.pi, shape)
    return (p - 2 * np.pi * np.round(p / (2 * np.pi))).astype(np.float32)


@pytest.mark.parametrize("W", [3, 4, 5, 8, 9, 10, 15, 16, 17, 31, 32, 33, 48, 59, 60, 61])
@pytest.mark.parametrize("H", [3, 33, 64, 500])
def test_few_columns(ctx, orc, H, W):
    """Widths around the words of 16 pixels, the rings that fit (W / 2) and the last width of this path, heights below and
    above the 1024 pixels that a wavefront lists at a time; three maps in a call, from sparse to the densest residues."""
    rng = np.random.default_rng(1000 * H + W)
    for noise in (0.5, 0.6, 0.8, 1.0):
        _equal(ctx, orc, _noisy(rng, (3, H, W), noise))


@pytest.mark.parametrize("W", [20, 60])
def test_far_and_unreachable_charges(ctx, orc, W):
    """Vortices of one sign far from each other and from the borders: scans that go past the first 64 positions, and
    ones that end without a hit (a residue in the middle column, with the largest ring short of both borders)."""
    H = 400
    y, x = np.mgrid[0:H, 0:W].astype(np.float64)
    phi = np.zeros((H, W))
    for i, cx in enumerate((W // 2 - 0.5, W // 2 - 0.5, W // 3 + 0.5, W // 2 + 0.5, W // 2 - 0.5)):
        phi += np.arctan2(y - (40.5 + 75 * i), x - cx)
    w = np.angle(np.exp(1j * phi)).astype(np.float32)[None]
    assert (_equal(ctx, orc, w) != 0).sum() >= 5


def test_tall_map_time(ctx):
    """One 2000 x 24 map of dense residues: about 100 ns a residue in all, and 206 when its rows ran side by side; the
    bound lies between."""
    w = torch.from_numpy(_noisy(np.random.default_rng(5), (1, 2000, 24), 0.8)).cuda()
    n = int((ctx.goldstein(w)[0] != 0).sum())
    spent = []
    for _ in range(20):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        ctx.goldstein(w)
        torch.cuda.synchronize()
        spent.append(time.perf_counter() - t0)
    print(f"{n} residues, {np.median(spent) * 1e9 / n:.0f} ns each")
    assert np.median(spent) < 150e-9 * n
