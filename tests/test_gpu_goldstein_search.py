"""The level search of the Goldstein fill on large maps: maps whose cuts leave a loop of free pixels with a non-zero sum of
steps, so that the 2 pi counts depend on the path and the spanning forest hands over to the search, against the host
specification (integers, so bit for bit)."""
import numpy as np
import pytest
import torch

import ctdm_amd

START_ROW = 20  # the fill starts in the middle of this row (or diagonally down and left from there, where that is cut)


def _map(H, W):
    """A slope with one noisy patch of 512 x 512, whose seed was found by trying (about one in 300 leaves such a loop)."""
    y, x = np.mgrid[0:H, 0:W]
    p = 0.11 * x + 0.07 * y
    p[100:612, 300:812] += np.random.default_rng(54).uniform(-0.7 * np.pi, 0.7 * np.pi, (512, 512))
    return np.angle(np.exp(1j * p)).astype(np.float32)


def _inconsistent_edges(w, cuts, k):
    """Edges between reached free pixels whose counts differ by another number than the edge's own step."""
    free = (cuts == 0) & (k != -2 ** 31)
    kk, n = k.astype(np.int64), 0
    for ax in (0, 1):
        lo, hi = [slice(None)] * 2, [slice(None)] * 2
        lo[ax], hi[ax] = slice(None, -1), slice(1, None)
        lo, hi = tuple(lo), tuple(hi)
        step = np.rint((w[hi] - w[lo]) * np.float32(0.15915494309189533577)).astype(np.int64)
        n += int(((kk[hi] - kk[lo] != -step) & free[hi] & free[lo]).sum())
    return n


def _levels(cuts):
    """(number of levels, largest level) of the search from its start pixel."""
    H, W = cuts.shape
    open_ = np.zeros((H + 2, W + 2), bool)
    open_[1:-1, 1:-1] = cuts == 0
    y, x = START_ROW, W // 2
    while not open_[y + 1, x + 1]:
        y, x = y + 1, x - 1
    flat, pitch = open_.reshape(-1), W + 2
    level = np.array([(y + 1) * pitch + x + 1])
    flat[level] = False
    depth = most = 0
    while len(level):
        depth, most = depth + 1, max(most, len(level))
        level = np.unique(np.concatenate([level + d for d in (1, -1, pitch, -pitch)]))
        level = level[flat[level]]
        flat[level] = False
    return depth, most


CASES = [(1264, 1020), (1024, 1024), (700, 1500)]


@pytest.mark.parametrize("H, W", CASES)
def test_inputs_need_the_search(orc, H, W):
    """Each map has an inconsistent loop and parent chains of over a thousand pixels; the first one's levels are larger than
    the 327 queue entries that its cut bits leave in 160 KiB of LDS."""
    w = _map(H, W)
    _, cuts, k, _ = (a[0] for a in orc.goldstein(w[None]))
    assert _inconsistent_edges(w, cuts, k) > 0
    depth, most = _levels(cuts)
    print(f"{H} x {W}: {depth} levels, largest {most}")
    assert depth > 1000
    if H * W > 1280000:
        assert most > 327


@pytest.mark.gpu
@pytest.mark.parametrize("H, W", CASES)
def test_large_inconsistent_maps(ctx, orc, H, W):
    """Alone and between two maps that take the forest."""
    smooth = np.angle(np.exp(1j * (0.11 * np.arange(W)[None] + 0.07 * np.arange(H)[:, None]))).astype(np.float32)
    w = np.stack([smooth, _map(H, W), smooth])
    for maps in (w[1:2], w):
        got = [t.cpu().numpy() for t in ctx.goldstein(torch.from_numpy(maps).cuda())]
        for name, g, r in zip(("residues", "cuts", "k2pi", "unwrapped"), got, orc.goldstein(maps)):
            assert np.array_equal(g.view(np.uint32) if g.dtype == np.float32 else g,
                                  r.view(np.uint32) if r.dtype == np.float32 else r), name
