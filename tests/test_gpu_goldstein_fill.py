"""The Goldstein fill without a search (spanning forest over 64 x 32 tiles, joined across their borders) and its fallback,
against the host specification's breadth-first search: 2 pi counts are whole numbers and the phases follow from them, so
every output must be equal bit for bit (tolerance zero)."""
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
    return ref


def _noisy(rng, shape, noise):
    B, H, W = shape
    y, x = np.mgrid[0:H, 0:W]
    p = 0.11 * x + 0.07 * y + 25 * ((x / W - 0.5) ** 2 + (y / H - 0.4) ** 2)
    return np.angle(np.exp(1j * (p + noise * rng.standard_normal(shape)))).astype(np.float32)


@pytest.mark.parametrize("H", [3, 31, 32, 33, 65])
@pytest.mark.parametrize("W", [4, 63, 64, 65, 129, 200])
def test_tile_edges(ctx, orc, H, W):
    """Maps that end at, one before and one after a tile border, with no cut, a few, and enough to break the map into
    many components; three maps in a call (odd map sizes leave the second and third at odd offsets)."""
    rng = np.random.default_rng(1000 * H + W)
    for noise in (0.0, 0.8, 1.5):
        _equal(ctx, orc, _noisy(rng, (3, H, W), noise))


def test_winding_paths(ctx, orc):
    """Walls of phase noise that leave corridors through many tiles in turn, against the raster order and with it."""
    rng = np.random.default_rng(2)
    w = _noisy(rng, (2, 260, 330), 0.2)
    for i in range(8):  # horizontal walls with a gap at alternating ends
        y = 30 * (i + 1)
        w[0, y:y + 6, (20 if i % 2 else 0):(330 if i % 2 else 310)] = rng.uniform(-np.pi, np.pi, (6, 310))
    for i in range(10):
        x = 30 * (i + 1)
        w[1, (20 if i % 2 else 0):(260 if i % 2 else 240), x:x + 6] = rng.uniform(-np.pi, np.pi, (240, 6))
    _equal(ctx, orc, w)


def test_inconsistent_map_takes_the_search(ctx, orc):
    """A map whose cuts leave a loop of free pixels with a non-zero sum of steps (found by trying seeds): the counts depend
    on the path, and it takes the search's. Alone, and among maps that do not."""
    H = W = 128
    rng = np.random.default_rng(58)
    y, x = np.mgrid[0:H, 0:W] / W
    w = np.angle(np.exp(1j * (30 * ((x - .5) ** 2 + (y - .5) ** 2) + 0.65 * 1.9 * rng.standard_normal((64, H, W)))))
    w = w.astype(np.float32)[39:42]
    _, cuts, k, _ = _equal(ctx, orc, w)
    step = np.rint((w[1, :, 1:] - w[1, :, :-1]) * np.float32(0.15915494309189533577)).astype(np.int64)
    step_y = np.rint((w[1, 1:] - w[1, :-1]) * np.float32(0.15915494309189533577)).astype(np.int64)
    free = (cuts[1] == 0) & (k[1] != -2 ** 31)
    kk = k[1].astype(np.int64)
    bad = ((kk[:, 1:] - kk[:, :-1] != -step) & free[:, 1:] & free[:, :-1]).sum()
    bad += ((kk[1:] - kk[:-1] != -step_y) & free[1:] & free[:-1]).sum()
    assert bad > 0  # the map is one
    _equal(ctx, orc, w[1:2])
