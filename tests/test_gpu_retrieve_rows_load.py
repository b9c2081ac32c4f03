"""Row-wise retrieval's paired pixel loads: frames that start at any pixel of a buffer (no alignment beyond the pixel's own)
give the bits of the same frames at an aligned address, in every format and width, and the first column and last row, where
the resampling's positions meet the border, agree with the FP64 oracle.

Tolerance: uniform random frames; FP32 transforms of 18 stages leave 6e-8 sqrt(18) = 2.5e-7 of the row's rms, 5 sigma 1.3e-6. The
compared quantity is the complex ratio's phase where both moduli are at least a tenth of their rms (4 times that, 1e-5 each,
so 2e-5 for the difference of two); the bar is 4e-5."""
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


@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.float32])
@pytest.mark.parametrize("W", [256, 512, 1024])
def test_any_pixel_offset(ctx, dtype, W):
    rng = np.random.default_rng(W)
    frames = rng.integers(0, 256, (2, 2, W, W)).astype(dtype)
    center = W // 4
    ref = None
    for off in (0, 1, 3):
        dev = []
        for f in frames:
            raw = np.concatenate([np.zeros(off, dtype), f.reshape(-1)])
            dev.append(torch.from_numpy(raw).cuda()[off:].view(2, W, W))
        got = ctx.retrieve_rows(dev[0], dev[1], center)
        if ref is None:
            ref = got
        for a, b in zip(got, ref):
            assert torch.equal(a, b), off
    r = orc.retrieve_rows(frames[0, 1].astype(np.float32), frames[1, 1].astype(np.float32), center)
    d = np.abs(np.angle(np.exp(1j * (ref[0][1].cpu().numpy() - r["wrapped"]))))
    # moduli of the two fields, from the oracle's own transform of the resampled rows
    def modulus(img):
        N2 = W // 4
        i = np.arange(W) * (W - 1) / W
        j = np.arange(N2) * (W - 1) / N2
        ix, iy = i.astype(int), j.astype(int)
        a, b = i - ix, (j - iy)[:, None]
        g = img.astype(np.float64)
        top = g[iy][:, ix] * (1 - a) + g[iy][:, np.minimum(ix + 1, W - 1)] * a
        bot = g[iy + 1][:, ix] * (1 - a) + g[iy + 1][:, np.minimum(ix + 1, W - 1)] * a
        X = np.fft.fft(top * (1 - b) + bot * b, axis=1)
        k = (center + W // 2 + np.arange(-W // 8, W // 8)) % W
        return np.abs(np.fft.ifft(np.fft.ifftshift(X[:, k], axes=1), axis=1)).T
    ms, mb = modulus(frames[0, 1]), modulus(frames[1, 1])
    ok = (ms > 0.1 * np.sqrt((ms ** 2).mean())) & (mb > 0.1 * np.sqrt((mb ** 2).mean()))
    print(f"W={W} {np.dtype(dtype).name}: phase {d[ok].max():.1e} over {ok.mean():.2f} of the map")
    assert ok.mean() > 0.9 and d[ok].max() <= 4e-5
