"""The 3 x 3 median's instruction sequence for comparable values and its fallback with NaN, against the selection sort of
the specification (fifth pick, strict '<', first minimum kept; borders copied): the result is one of the inputs, so it must be
equal (tolerance zero; zeros of either sign count as equal)."""
import numpy as np
import pytest
import torch

import ctdm_amd

pytestmark = pytest.mark.gpu


def sort_median(m):
    out = m.copy()
    H, W = m.shape
    for y in range(1, H - 1):
        for x in range(1, W - 1):
            v = [m[y + dy, x + dx] for dx in (-1, 0, 1) for dy in (-1, 0, 1)]
            for i in range(5):
                mn = i
                for k in range(i + 1, 9):
                    if v[k] < v[mn]:
                        mn = k
                v[i], v[mn] = v[mn], v[i]
            out[y, x] = v[4]
    return out


@pytest.mark.parametrize("kind", ["random", "ties", "infinite", "nan", "extremes"])
def test_median_equals_the_sort(ctx, kind):
    rng = np.random.default_rng(len(kind))
    m = rng.standard_normal((2, 37, 53)).astype(np.float32)
    if kind == "ties":
        m = np.round(m)
    elif kind == "infinite":
        m[rng.uniform(size=m.shape) < 0.3] = np.inf
        m[rng.uniform(size=m.shape) < 0.3] = -np.inf
    elif kind == "nan":
        m[rng.uniform(size=m.shape) < 0.15] = np.nan
        m[0, 10:20, 10:20] = np.nan
    elif kind == "extremes":
        big = np.finfo(np.float32).max
        m = rng.choice(np.array([big, -big, 1e-45, -1e-45, 0.0], np.float32), m.shape)
    got = ctx.median3x3(torch.from_numpy(m).cuda()).cpu().numpy()
    for g, w in zip(got, m):
        assert np.array_equal(g, sort_median(w), equal_nan=True)
