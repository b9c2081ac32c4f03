"""Band widths around the column pass's tiles: rows of the band arrays are padded to eight columns, and few images take
the narrower tile. Against the FP64 oracle at widths whose last tile holds one column, a full tile, or all but one, for
one pair and for enough pairs to take the wide tile.

Tolerance: FP32 transforms of up to 28 stages leave about 6e-8 sqrt(28) = 3.2e-7 of the hologram's rms, 5.3 times the
sideband's modulus (200 of 1000), whose share in the band is radius / 512 of it at most: 5e-7 of a field of nearly
constant modulus, 2.5e-6 at 5 sigma and 3.5e-6 for the ratio of two. The bar is 2e-5 for float transcendentals on top."""
import numpy as np
import pytest
import torch

import ctdm_amd
from oracle import binding as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = ctdm_amd.Context()
    yield c
    c.close()


@pytest.mark.parametrize("H,M,radius,pairs", [(256, 64, 7, 1), (256, 64, 8, 24), (512, 128, 32, 1), (512, 128, 31, 20),
                                              (1024, 256, 60, 1), (1024, 256, 68, 6), (1024, 256, 0, 1)])
def test_band_widths(ctx, H, M, radius, pairs):
    rng = np.random.default_rng(radius + pairs)
    y, x = np.mgrid[0:H, 0:H]
    row, col = H // 2 + H // 4, H // 2 + H // 8
    carrier = 2 * np.pi * ((col - H // 2) * x + (row - H // 2) * y) / H
    low = np.cos(2 * np.pi * 2 * x / H) + np.sin(2 * np.pi * 3 * y / H)
    holo = np.stack([1000 + 400 * np.cos(carrier + 0.3 * k + 0.5 * low) for k in range(pairs)])
    holo = (holo + rng.standard_normal(holo.shape)).astype(np.float32)
    bg = np.stack([1000 + 400 * np.cos(carrier)] * pairs).astype(np.float32)
    crop = ctdm_amd.Crop(row, col, radius, M)
    ph, la = ctx.retrieve(torch.from_numpy(holo).cuda(), torch.from_numpy(bg).cuda(), crop)[:2]
    for k in {0, pairs - 1}:
        r = orc.retrieve(holo[k], bg[k], *crop.astuple())
        d = np.angle(np.exp(1j * (ph[k].cpu().numpy() - r["wrapped"])))
        e, ea = np.abs(d).max(), np.abs(la[k].cpu().numpy() - r["logamp"]).max()
        print(f"H={H} radius={radius} pair {k}: phase {e:.1e}, log-amplitude {ea:.1e}")
        assert e <= 2e-5 and ea <= 2e-5
