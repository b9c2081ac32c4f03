"""The Goldstein cut search's row pipeline (k_gs_pair) at the sizes and charge layouts where it can go wrong,
against the host specification: residues, cuts, 2 pi counts and unwrapped phases are whole-number work or single
rounded operations, so every output must be equal bit for bit (tolerance zero)."""
import numpy as np
import pytest
import torch

import ctdm_amd

pytestmark = pytest.mark.gpu


def _equal(ctx, orc, w):
    got = [t.cpu().numpy() for t in ctx.goldstein(torch.from_numpy(w).cuda())]
    ref = orc.goldstein(w)
    for name, g, r in zip(("residues", "cuts", "k2pi", "unwrapped"), got, ref):
        assert np.array_equal(g.view(np.uint32) if g.dtype == np.float32 else g,
                              r.view(np.uint32) if r.dtype == np.float32 else r), name
    return ref[0]


@pytest.mark.parametrize("H", [3, 5, 33, 35, 67])
@pytest.mark.parametrize("W", [3, 6, 7, 8, 9, 31, 32, 33, 64, 95])
def test_row_and_word_edges(ctx, orc, H, W):
    """Rows of fewer pixels than the rings reach, rows that end on either side of a 32-pixel word, and one row
    more or less than the rows in flight (32 interior rows); uniform random phase, three maps in a call (odd map
    sizes leave the second and third at odd addresses)."""
    rng = np.random.default_rng(100 * H + W)
    res = _equal(ctx, orc, rng.uniform(-np.pi, np.pi, size=(3, H, W)).astype(np.float32))
    assert H < 5 or W < 6 or (res != 0).any()


@pytest.mark.parametrize("dist", [4, 8, 13, 41, 60, 170])
@pytest.mark.parametrize("axis", [0, 1])
def test_far_partners(ctx, orc, dist, axis):
    """Vortex pairs `dist` pixels apart on a 180 x 400 map: partners on each side of the expected reach (40 at this
    density) and of four times it, so the map is searched in one, two and three attempts."""
    H, W = 180, 400
    y, x = np.mgrid[0:H, 0:W].astype(np.float64)
    phi = np.zeros((H, W))
    for k, (cx, cy) in enumerate([(110.5, 20.5), (150.5, 90.5)] if axis == 0 or dist < 100 else [(200.5, 4.5)]):
        ex, ey = (cx + dist, cy) if axis == 0 else (cx, cy + (dist if cy + dist < H - 2 else -dist if cy > dist else 60))
        s = 1.0 if k == 0 else -1.0
        phi += s * (np.arctan2(y - cy, x - cx) - np.arctan2(y - ey, x - ex))
    w = np.angle(np.exp(1j * phi)).astype(np.float32)[None]
    assert (_equal(ctx, orc, w) != 0).sum() >= 2


@pytest.mark.parametrize("shape,noise", [((2, 150, 211), 0.62), ((1, 96, 700), 0.56), ((2, 300, 64), 0.7)])
def test_densities(ctx, orc, shape, noise):
    """Residue densities on each side of the lines where the expected reach changes (0.25, 0.1 and 0.05)."""
    rng = np.random.default_rng(5)
    y, x = np.mgrid[0:shape[1], 0:shape[2]].astype(np.float64)
    v = 9.0 * np.exp(-((x - 40) ** 2 + (y - 50) ** 2) / 900.0) + 0.05 * x
    w = np.angle(np.exp(1j * (v + rng.uniform(-noise * np.pi, noise * np.pi, shape)))).astype(np.float32)
    assert (_equal(ctx, orc, w) != 0).any()


def test_one_sign_of_charge(ctx, orc):
    """Charges of one sign only, far from every border: no opposite charge, each scan ends at a border."""
    H, W = 120, 150
    y, x = np.mgrid[0:H, 0:W].astype(np.float64)
    phi = sum(np.arctan2(y - cy, x - cx) for cx, cy in [(60.5, 50.5), (80.5, 60.5), (75.5, 51.5)])
    w = np.angle(np.exp(1j * phi)).astype(np.float32)[None]
    assert (_equal(ctx, orc, w) != 0).sum() >= 3
