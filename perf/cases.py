"""Performance cases of the reconstruction path: what its users run, through the public entry points.

A case is a dict of plain values with a "kind":

  frames     retrieve (2-D sideband crop) + unwrap_dct of a stack of hologram pairs
  rows       retrieve_rows (row-wise retrieval) + unwrap_dct
  goldstein  branch-cut unwrapping of wrapped maps of any size
  adjoint    unwrap_dct, its adjoint, and the gather (adjoint of the Ewald scatter)
  maps       recon_from_maps: saved phase and amplitude maps -> volume
  steps      the reconstruction call by call: spectra, scatter, normalisation, 3-D FFT, positivity loop
  fit        fit_pgd on measured spectra
  cells      reconstruct: one or more cells of hologram pairs -> volumes, in one captured graph

Inputs are seeded and made on the GPU: a phantom of 3-D Gaussian bodies seen along tilted directions, its
projected phase and absorption, and off-axis holograms of it with a carrier near a quarter of the sampling
rate, sensor noise, and 8- or 16-bit quantisation where the case says so. One context serves all calls, as
in a program that keeps one per device.
"""
import math

import numpy as np
import torch

import ctdm_amd

DEV = "cuda"
WAVELENGTH, N_MED, PIXEL = 532e-9, 1.337, 0.1e-6
FAST = ctdm_amd.UNWRAP_SINCOS | ctdm_amd.UNWRAP_CONGRUENT
FULL_SCALE = {"u8": 255.0, "u16": 4095.0}

_ctx = None


def _context():
    global _ctx
    if _ctx is None:
        _ctx = ctdm_amd.Context(0)
    return _ctx


# ---------------------------------------------------------------- cases
def listed():
    return [
        # live preview: one binned 8-bit camera frame against its background; launches and latency
        dict(name="frame_256_u8", kind="frames", batch=1, H=256, M=64, px="u8", fast=False),
        # the single-hologram workload: one full frame
        dict(name="frame_1024", kind="frames", batch=1, H=1024, M=256, px="f32", fast=False),
        # the front end of one cell: all illumination angles of a full-size acquisition
        dict(name="angles_60x1024", kind="frames", batch=60, H=1024, M=256, px="f32", fast=False),
        # the default (row-wise) retrieval with the sin/cos unwrapping on 16-bit half-size frames
        dict(name="rows_45x512_u16", kind="rows", batch=45, H=512, px="u16", fast=True),
        # per-frame branch-cut unwrapping of one retrieved map, moderate noise
        dict(name="goldstein_frame", kind="goldstein", batch=1, H=256, W=256, noise=0.6),
        # the branch-cut benchmark: a stack of noisy maps, dense residues
        dict(name="goldstein_64x512", kind="goldstein", batch=64, H=512, W=512, noise=0.8),
        # gradients through the unwrapping and the Ewald sampling, for a program that trains or fits
        dict(name="adjoint_24x192", kind="adjoint", A=24, V=192, sincos=True),
        # reload of a saved acquisition: median, sanitising and logarithm of the maps, then the volume
        dict(name="maps_45_128", kind="maps", A=45, V=128, iters=10),
        # the reconstruction written out call by call
        dict(name="steps_30_192", kind="steps", A=30, V=192, iters=10),
        # the projected-gradient fit: 120 angles, 50 steps
        dict(name="fit_120_256", kind="fit", A=120, V=256, iters=50, step=1.0),
        # the headline cell: 60 x 1024^2 float32 pairs -> 256^3, 10 iterations
        dict(name="cell_60x1024_256", kind="cells", cells="60:1024:256", px="f32", iters=10),
        # eight uneven cells of 8-bit frames in one graph
        dict(name="cells_uneven_u8", kind="cells",
             cells="30:1024:128,45:1024:192,60:1024:256,60:1024:128,90:1024:192,90:1024:256,120:1024:128,120:1024:192",
             px="u8", iters=10),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["frames", "rows", "goldstein", "adjoint", "maps", "steps", "fit", "cells"])
    px = rng.choice(["f32", "u8", "u16"])
    if kind == "frames":
        H, M = rng.choice([(256, 64), (256, 32), (512, 128), (512, 64), (1024, 256), (1024, 192), (1024, 128)])
        return dict(kind=kind, batch=_log_int(rng, 1, 64), H=H, M=M, px=px, fast=rng.random() < 0.5)
    if kind == "rows":
        return dict(kind=kind, batch=_log_int(rng, 1, 64), H=rng.choice([256, 512, 1024]), px=px,
                    fast=rng.random() < 0.5)
    if kind == "goldstein":
        return dict(kind=kind, batch=_log_int(rng, 1, 48), H=_log_int(rng, 48, 520), W=_log_int(rng, 48, 520),
                    noise=round(rng.uniform(0.3, 0.8), 2))
    V = rng.choice([64, 128, 192, 256])
    A = _log_int(rng, 3, 90)
    if kind == "adjoint":
        return dict(kind=kind, A=A, V=V, sincos=rng.random() < 0.5)
    if kind in ("maps", "steps"):
        return dict(kind=kind, A=A, V=V, iters=rng.randint(1, 15))
    if kind == "fit":
        return dict(kind=kind, A=A, V=V, iters=rng.randint(3, 30), step=rng.choice([0.5, 1.0]))
    cells = []
    for _ in range(rng.randint(1, 4)):
        H, V = rng.choice([(256, 64), (512, 128), (1024, 128), (1024, 192), (1024, 256)])
        cells.append("%d:%d:%d" % (_log_int(rng, 4, 70), H, V))
    return dict(kind=kind, cells=",".join(cells), px=px, iters=rng.randint(2, 12))


def _cells_of(case):
    return [tuple(int(x) for x in c.split(":")) for c in case["cells"].split(",")]


# ---------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 2654435761 % (1 << 62) + 17)


def _uniform(g, *shape, lo=0.0, hi=1.0):
    return lo + (hi - lo) * torch.rand(*shape, generator=g, device=DEV)


def _cone(seed, A):
    """A illumination angles on a cone of illumination NA 1.0, azimuth offset and jitter by the seed."""
    r = np.random.RandomState(int(seed) % (1 << 31))
    az = 2 * np.pi * (np.arange(A) + r.uniform(0, 1) + 0.1 * r.uniform(-1, 1, A)) / max(A, 1)
    s = (1.0 / N_MED) * (1 + 0.02 * r.uniform(-1, 1, A))
    return np.stack([np.arcsin(s * np.sin(az)), np.arcsin(s * np.cos(az))], axis=1)


def _bodies(g, H):
    """Gaussian bodies in units of pixels of an H x H frame: centre (3), sigma, phase peak."""
    K = 7
    c = _uniform(g, K, 3, lo=-0.12, hi=0.12) * H
    s = torch.cat([_uniform(g, 2, lo=0.08, hi=0.12), _uniform(g, K - 2, lo=0.02, hi=0.04)]) * H
    p = torch.cat([_uniform(g, 2, lo=1.5, hi=3.0), _uniform(g, K - 2, lo=0.2, hi=0.6)])
    c[:2] *= 0.3
    return c, s, p


def _maps(g, H, angles):
    """Projected phase and log-amplitude, A x H x H float32, for the given directions."""
    c, s, p = _bodies(g, H)
    d = torch.as_tensor(np.tan(np.clip(angles, -1.0, 1.0)), dtype=torch.float32, device=DEV)
    grid = torch.arange(H, device=DEV, dtype=torch.float32) - H / 2
    cx = c[None, :, 0] - d[:, 0:1] * c[None, :, 2]
    cy = c[None, :, 1] - d[:, 1:2] * c[None, :, 2]
    ex = torch.exp(-((grid[None, None] - cx[..., None]) / s[None, :, None]) ** 2 / 2)  # A, K, H
    ey = torch.exp(-((grid[None, None] - cy[..., None]) / s[None, :, None]) ** 2 / 2) * p[None, :, None]
    phase = torch.bmm(ey.transpose(1, 2).contiguous(), ex)
    return phase, -0.25 - 0.06 * phase  # the sample is darker than the background all over


def _carrier(seed, H):
    """Carrier frequency (x, y) in cycles per pixel, within a quarter of a bin of a bin's centre."""
    r = np.random.RandomState((int(seed) * 7 + 3) % (1 << 31))
    k = H // 4 + r.randint(-(H // 64), H // 64 + 1, 2) + r.uniform(-0.25, 0.25, 2)
    return k[0] / H, k[1] / H


def _quantise(x, px):
    if px == "f32":
        return x
    top = FULL_SCALE[px]
    q = (x * (top / 4.6)).round_().clamp_(0, top)
    return q.to(torch.uint8) if px == "u8" else q.to(torch.int16).view(torch.uint16)


def _holograms(seed, A, H, px, angles):
    """(holo, bg), A x H x H: I = 1 + a^2 + 2 a cos(2 pi (fx x + fy y) + phase) + noise."""
    g = _gen(seed)
    fx, fy = _carrier(seed, H)
    x = torch.arange(H, device=DEV, dtype=torch.float32)
    carrier = 2 * math.pi * (((fx * x)[None, :] + (fy * x)[:, None]) % 1.0)
    dt = {"f32": torch.float32, "u8": torch.uint8, "u16": torch.uint16}[px]
    holo = torch.empty((A, H, H), dtype=dt, device=DEV)
    bg = torch.empty((A, H, H), dtype=dt, device=DEV)
    phase_all = _maps(g, H, angles)
    for a in range(A):
        ph, la = phase_all[0][a], phase_all[1][a]
        amp = torch.exp(la)
        noise = torch.randn(2, H, H, generator=g, device=DEV) * 0.01
        holo[a] = _quantise((1.3 + amp * amp + 2 * amp * torch.cos(carrier + ph) + noise[0]).clamp_(0, 4.6), px)
        bg[a] = _quantise((2.3 + 2 * torch.cos(carrier) + noise[1]).clamp_(0, 4.6), px)
    return holo, bg


def _crop(seed, H, M):
    fx, fy = _carrier(seed, H)
    row, col = H // 2 + int(round(fy * H)), H // 2 + int(round(fx * H))
    return ctdm_amd.Crop(row, col, abs(row - H // 2) // 3, M)


def _wrapped(seed, batch, H, W, noise):
    """Wrapped maps: 8 Gaussians of up to 40 rad plus uniform noise in +-noise*pi."""
    g = _gen(seed)
    k = 8
    peak = _uniform(g, batch, k, lo=-40.0, hi=40.0)
    cx, cy = _uniform(g, batch, k) * W, _uniform(g, batch, k) * H
    s = _uniform(g, batch, k, lo=20.0, hi=80.0)
    x = torch.arange(W, device=DEV, dtype=torch.float32)
    y = torch.arange(H, device=DEV, dtype=torch.float32)
    ex = torch.exp(-((x - cx[..., None]) / s[..., None]) ** 2 / 2)
    ey = torch.exp(-((y - cy[..., None]) / s[..., None]) ** 2 / 2) * peak[..., None]
    v = torch.bmm(ey.transpose(1, 2).contiguous(), ex)
    v += _uniform(g, batch, H, W, lo=-noise * math.pi, hi=noise * math.pi)
    return v - 2 * math.pi * torch.round(v / (2 * math.pi))


def _optics(V):
    return ctdm_amd.optics_for(V)


def _map_stack(seed, A, V):
    """Unwrapped phase and log-amplitude maps (A x V x V) of a cell, with pixel noise, and the angles."""
    ang = _cone(seed, A)
    g = _gen(seed)
    ph, la = _maps(g, V, ang)
    ph = ph + 0.01 * torch.randn(A, V, V, generator=g, device=DEV)
    la = la + 0.005 * torch.randn(A, V, V, generator=g, device=DEV)
    return ph.contiguous(), la.contiguous(), ang


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case, "seed": seed, "ctx": _context()}
    if kind in ("frames", "rows"):
        A, H = case["batch"], case["H"]
        st["holo"], st["bg"] = _holograms(seed, A, H, case["px"], _cone(seed, A))
        st["crop"] = _crop(seed, H, case.get("M", H // 4))
        st["flags"] = FAST if case["fast"] else 0
    elif kind == "goldstein":
        st["wrapped"] = _wrapped(seed, case["batch"], case["H"], case["W"], case["noise"])
    elif kind == "adjoint":
        A, V = case["A"], case["V"]
        ph, la, st["angles"] = _map_stack(seed, A, V)
        ph = ph * 2.5
        st["wrapped"] = ph - 2 * math.pi * torch.round(ph / (2 * math.pi))
        g = _gen(seed + 1)
        res = torch.randn(A, V, V, generator=g, device=DEV)  # a fit's residual: noise without its smooth part
        smooth = torch.nn.functional.avg_pool2d(res[:, None], 8)
        st["grad"] = (res - torch.nn.functional.interpolate(smooth, scale_factor=8)[:, 0]).contiguous()
        st["F"] = torch.view_as_complex(torch.randn(V, V, V, 2, generator=g, device=DEV))
        st["flags"] = ctdm_amd.UNWRAP_SINCOS if case["sincos"] else 0
        st["optics"] = _optics(V)
    elif kind == "maps":
        st["phase"], la, st["angles"] = _map_stack(seed, case["A"], case["V"])
        st["amp"] = torch.exp(la)
        st["optics"] = _optics(case["V"])
    elif kind == "steps":
        st["phase"], st["logamp"], st["angles"] = _map_stack(seed, case["A"], case["V"])
        st["optics"] = _optics(case["V"])
    elif kind == "fit":
        A, V = case["A"], case["V"]
        ph, la, st["angles"] = _map_stack(seed, A, V)
        st["optics"] = _optics(V)
        st["spec"] = _rytov(ph, la)
        F, hits = _scatter(st["spec"], st["angles"], V, st["optics"])
        st["f0"] = torch.fft.ifftn(F / hits.clamp(min=1.0) / st["optics"].dx).contiguous()
    else:
        st["cells"] = []
        for i, (A, H, V) in enumerate(_cells_of(case)):
            ang = _cone(seed + 100 * i, A)
            holo, bg = _holograms(seed + 100 * i, A, H, case["px"], ang)
            st["cells"].append(dict(holo=holo, bg=bg, angles=ang, V=V, iters=case["iters"],
                                    optics=ctdm_amd.optics_for(V, H),
                                    ri=torch.empty((V, V, V), dtype=torch.complex64, device=DEV)))
    return st


# ---------------------------------------------------------------- one pass
def run(st):
    case, ctx = st["case"], st["ctx"]
    kind = case["kind"]
    if kind == "frames":
        wrapped, logamp = ctx.retrieve(st["holo"], st["bg"], st["crop"])
        return {"logamp": logamp, "unwrapped": ctx.unwrap_dct(wrapped, st["flags"])}
    if kind == "rows":
        wrapped, logamp = ctx.retrieve_rows(st["holo"], st["bg"], st["crop"].col)
        return {"logamp": logamp, "unwrapped": ctx.unwrap_dct(wrapped, st["flags"])}
    if kind == "goldstein":
        res, cuts, k, un = ctx.goldstein(st["wrapped"])
        return {"residues": res, "cuts": cuts, "k": k, "unwrapped": un}
    if kind == "adjoint":
        un = ctx.unwrap_dct(st["wrapped"], st["flags"])
        gw = ctx.unwrap_dct_adjoint(st["wrapped"], st["grad"], st["flags"])
        spec = ctx.ewald_gather(st["F"], st["angles"], case["V"], st["optics"])
        return {"unwrapped": un, "grad": gw, "spec": spec}
    if kind == "maps":
        return {"ri": ctx.recon_from_maps(st["phase"], st["amp"], st["angles"], st["optics"], case["iters"],
                                          ctdm_amd.MAPS_MEDIAN | ctdm_amd.MAPS_AMPLITUDE)}
    if kind == "steps":
        V, o = case["V"], st["optics"]
        spec = ctx.rytov_spectrum(st["phase"], st["logamp"])
        F, hits = ctx.ewald_scatter(spec, st["angles"], V, o)
        meas = ctx.normalize_measured(F, hits, o.dx)
        f = ctx.fft3d(F, +1)
        return {"spec": spec, "hits": hits, "meas": meas, "ri": ctx.positivity(f, meas, hits, case["iters"], o)}
    if kind == "fit":
        return {"ri": ctx.fit_pgd(st["f0"].clone(), st["spec"], st["angles"], st["optics"], case["iters"],
                                  case["step"])}
    ctx.reconstruct(st["cells"], mode=1, graph=True)
    return {"ri": [c["ri"] for c in st["cells"]],
            "crop": [v for c in st["cells"] for v in (c["crop_used"].row, c["crop_used"].col)]}


# ---------------------------------------------------------------- the least work of a pass
def _fft(n, per=1.0):
    return 5.0 * n * math.log2(n) * per


def _retrieval_work(A, H, M, px):
    b = {"f32": 4, "u8": 1, "u16": 2}[px]
    return dict(bytes=2.0 * A * H * H * b, flops=2.0 * A * (0.5 * _fft(H * H) + _fft(M * M)))


def _unwrap_flops(A, M):
    return A * (2 * 0.5 * _fft(M * M) + 15.0 * M * M)


def _volume_flops(A, V, iters):
    return A * _fft(V * V) + 10.0 * A * V * V + (2 * iters + 1) * _fft(V ** 3) + 30.0 * iters * V ** 3


def work(case):
    kind = case["kind"]
    if kind in ("frames", "rows"):
        M = case.get("M", case["H"] // 4)
        w = _retrieval_work(case["batch"], case["H"], M, case["px"])
        return dict(bytes=w["bytes"] + 3 * 4.0 * case["batch"] * M * M, flops=w["flops"] + _unwrap_flops(case["batch"], M))
    if kind == "goldstein":
        n = 1.0 * case["batch"] * case["H"] * case["W"]
        return dict(bytes=14.0 * n, flops=60.0 * n)
    A, V, n = case.get("A"), case.get("V"), 1.0 * case.get("A", 0) * case.get("V", 0) ** 2
    if kind == "adjoint":
        return dict(bytes=4 * 4.0 * n + 8.0 * min(n, V ** 3) + 8.0 * n, flops=2 * _unwrap_flops(A, V) + 40.0 * n)
    if kind == "maps":
        return dict(bytes=8.0 * n + 8.0 * V ** 3, flops=_volume_flops(A, V, case["iters"]) + 60.0 * n)
    if kind == "steps":
        return dict(bytes=8.0 * n + 8.0 * n + 20.0 * V ** 3, flops=_volume_flops(A, V, case["iters"]))
    if kind == "fit":
        return dict(bytes=8.0 * n + 16.0 * V ** 3, flops=_volume_flops(0, V, case["iters"]) + 20.0 * n)
    total = dict(bytes=0.0, flops=0.0)
    for A, H, V in _cells_of(case):
        w = _retrieval_work(A, H, V, case["px"])
        total["bytes"] += w["bytes"] + 8.0 * V ** 3
        total["flops"] += w["flops"] + _unwrap_flops(A, V) + _volume_flops(A, V, case["iters"])
    return total


# ---------------------------------------------------------------- the same in 64 bits, from the definitions
def _pixels(x):
    return x.view(torch.int16).double() if x.dtype == torch.uint16 else x.double()


def _combine(sp, bg):
    z = sp * bg.conj()
    return torch.atan2(z.imag, z.real), 0.5 * (torch.log(sp.abs() ** 2) - torch.log(bg.abs() ** 2))


def _retrieve64(holo, bg, row, col, radius, M):
    H = holo.shape[-1]
    lo, hi = max(-M // 2, -radius), min(M // 2 - 1, radius)
    q = torch.arange(lo, hi + 1, device=DEV)
    ry, cx = (row - H // 2 + q) % H, (col - H // 2 + q) % H

    def field(img):
        F = torch.fft.fft2(_pixels(img))
        S = torch.zeros(F.shape[0], M, M, dtype=F.dtype, device=DEV)
        S[:, (q % M)[:, None], (q % M)[None, :]] = F[:, ry[:, None], cx[None, :]]
        return torch.fft.ifft2(S)

    out = [_combine(field(holo[a:a + 8]), field(bg[a:a + 8])) for a in range(0, holo.shape[0], 8)]
    return torch.cat([o[0] for o in out]), torch.cat([o[1] for o in out])


def _retrieve_rows64(holo, bg, center):
    H = W = holo.shape[-1]
    N2, M = H // 4, W // 4
    i, j = torch.arange(W, device=DEV), torch.arange(N2, device=DEV)
    xs, ys = i * ((W - 1) / W), j * ((H - 1) / N2)
    ix, iy = xs.long(), ys.long()
    a, b = (xs - ix), (ys - iy)[:, None]
    d = torch.arange(M, device=DEV)
    d = torch.where(d < M // 2, d, d - M)

    def field(img):
        p = torch.nn.functional.pad(_pixels(img), (0, 1, 0, 1))
        t1 = p[:, iy][:, :, ix] * (1 - a) + p[:, iy][:, :, ix + 1] * a
        t2 = p[:, iy + 1][:, :, ix] * (1 - a) + p[:, iy + 1][:, :, ix + 1] * a
        X = torch.fft.fft(t1 * (1 - b) + t2 * b, dim=-1)
        return torch.fft.ifft(X[..., (center + W // 2 + d) % W], dim=-1).transpose(1, 2)

    out = [_combine(field(holo[k:k + 8]), field(bg[k:k + 8])) for k in range(0, holo.shape[0], 8)]
    return torch.cat([o[0] for o in out]), torch.cat([o[1] for o in out])


def _poisson64(rho):
    N = rho.shape[-1]
    n = torch.arange(N, device=DEV, dtype=torch.float64)
    D = torch.cos(math.pi * (2 * n[None, :] + 1) * n[:, None] / (2 * N)) * math.sqrt(2.0 / N)
    D[0] = math.sqrt(1.0 / N)
    e = torch.sin(math.pi * n / (2 * N)) ** 2
    lam = -4.0 * (e[:, None] + e[None, :])
    lam[0, 0] = 1.0
    X = torch.matmul(torch.matmul(D, rho), D.t().contiguous()) / lam
    X[..., 0, 0] = 0.0
    return torch.matmul(torch.matmul(D.t().contiguous(), X), D)


def _diffs(w):
    return w[..., :, 1:] - w[..., :, :-1], w[..., 1:, :] - w[..., :-1, :]


def _div(gx, gy, like):
    r = torch.zeros_like(like)
    r[..., :, :-1] += gx
    r[..., :, 1:] -= gx
    r[..., :-1, :] += gy
    r[..., 1:, :] -= gy
    return r


def _unwrap64(w, flags):
    gx, gy = _diffs(w)
    if flags & ctdm_amd.UNWRAP_SINCOS:
        gx, gy = torch.sin(gx), torch.sin(gy)
    else:
        gx, gy = (g - 2 * math.pi * torch.round(g / (2 * math.pi)) for g in (gx, gy))
    v = _poisson64(_div(gx, gy, w))
    if flags & ctdm_amd.UNWRAP_CONGRUENT:
        v = w + 2 * math.pi * torch.round((v - w) / (2 * math.pi))
    return v


def _adjoint64(w, g, flags):
    v = _poisson64(g)
    vx, vy = _diffs(v)
    if flags & ctdm_amd.UNWRAP_SINCOS:
        wx, wy = _diffs(w)
        vx, vy = vx * torch.cos(wx), vy * torch.cos(wy)
    return _div(vx, vy, v)


def _rytov(phase, logamp):
    """Rytov spectra of the maps, in their precision: (-1)^(kx + ky) times the transposed 2-D DFT."""
    M = phase.shape[-1]
    s = 1.0 - 2.0 * (torch.arange(M, device=DEV) % 2).to(phase.dtype)
    U = torch.fft.fft2(torch.complex(logamp, phase))
    return (U * (s[:, None] * s[None, :])).transpose(1, 2).contiguous()


def _caps(angles, V, o):
    """Per angle: (voxel plane index z, weight 4 pi f_z, on the cap) of every spectrum pixel [y][x]."""
    fm0 = o.n_med / o.wavelength
    df = 1.0 / (V * o.dx)
    k = torch.arange(V, device=DEV, dtype=torch.float64)
    k = torch.where(k < V // 2, k, k - V)
    for ax, ay in np.asarray(angles):
        fx0, fy0 = fm0 * math.sin(ay), fm0 * math.sin(ax)
        s0 = fm0 * fm0 - fx0 * fx0 - fy0 * fy0
        fx, fy = (k * df + fx0)[None, :], (k * df + fy0)[:, None]
        s = fm0 * fm0 - (fx * fx + fy * fy)
        ok = ~(s < 0) & (s0 >= 0)
        fz = torch.sqrt(s.clamp(min=0))
        q = (fz - math.sqrt(max(s0, 0.0))) / df
        nz = torch.where(q > 0, torch.floor(q + 0.5), torch.ceil(q - 0.5)).long() % V
        yield nz, 4 * math.pi * fz, ok


def _scatter(spec, angles, V, o):
    """Sum of 4 pi i f_z spec on the caps, and the hit counts, angle after angle, in spec's precision."""
    F = torch.zeros(V, V * V, dtype=spec.dtype, device=DEV)
    hits = torch.zeros(V, V * V, dtype=spec.real.dtype, device=DEV)
    p = torch.arange(V * V, device=DEV)
    for a, (nz, w, ok) in enumerate(_caps(angles, V, o)):
        w = (w * ok).to(hits.dtype).reshape(-1)
        at = (nz.reshape(-1), p)
        F[at] += 1j * w * spec[a].reshape(-1)
        hits[at] += ok.to(hits.dtype).reshape(-1)
    return F.view(V, V, V), hits.view(V, V, V)


def _est_n64(f, o):
    k2 = (2 * math.pi * o.n_med / o.wavelength) ** 2
    z = 1.0 - f / k2
    r = torch.sqrt(z)
    im = torch.where(z.imag == 0, torch.zeros_like(r.imag), r.imag)
    return torch.complex((r.real * o.n_med).clamp(min=o.n_med), (im * o.n_med).clamp(min=0.0))


def _modify64(n, o):
    k2 = (2 * math.pi * o.n_med / o.wavelength) ** 2
    return -k2 * ((n / o.n_med) ** 2 - 1.0)


def _loop64(f, meas, hits, iters, o, step=1.0):
    """n after `iters` iterations, octant-shifted."""
    n = _est_n64(f, o)
    for _ in range(iters):
        F = torch.fft.fftn(_modify64(n, o))
        F = torch.where(hits > 0, F + step * (meas - F), F)
        n = _est_n64(torch.fft.ifftn(F), o)
    return torch.fft.fftshift(n)


def _volume64(phase, logamp, angles, o, iters):
    V = phase.shape[-1]
    F, hits = _scatter(_rytov(phase, logamp), angles, V, o)
    meas = F / hits.clamp(min=1.0) / o.dx
    return _loop64(torch.fft.ifftn(meas), meas, hits, iters, o)


def _median64(x):
    y = x.double()
    out = y.clone()
    win = y.unfold(1, 3, 1).unfold(2, 3, 1).reshape(y.shape[0], y.shape[1] - 2, y.shape[2] - 2, 9)
    out[:, 1:-1, 1:-1] = win.median(dim=-1).values
    return out


def _search64(bg0):
    H = bg0.shape[-1]
    S = torch.fft.fftshift(torch.fft.fft2(_pixels(bg0))).abs()
    start = 600 * H // 1024
    at = start * H + int(S[start:].argmax())
    return at // H, at % H


def exact(case, seed):
    kind = case["kind"]
    if kind == "goldstein":  # whole numbers, and sums that follow from them
        return None
    st = prepare(case, seed)
    if kind in ("frames", "rows"):
        c = st["crop"]
        w, la = (_retrieve64(st["holo"], st["bg"], c.row, c.col, c.radius, c.M) if kind == "frames"
                 else _retrieve_rows64(st["holo"], st["bg"], c.col))
        return {"logamp": la, "unwrapped": _unwrap64(w, st["flags"])}
    if kind == "adjoint":
        A, V = case["A"], case["V"]
        w, F = st["wrapped"].double(), st["F"].to(torch.complex128).view(V, V * V)
        p = torch.arange(V * V, device=DEV)
        spec = torch.stack([(-1j * wt.reshape(-1) * ok.reshape(-1) * F[nz.reshape(-1), p]).view(V, V)
                            for nz, wt, ok in _caps(st["angles"], V, st["optics"])])
        return {"unwrapped": _unwrap64(w, st["flags"]), "grad": _adjoint64(w, st["grad"].double(), st["flags"]),
                "spec": spec}
    if kind == "maps":
        return {"ri": _volume64(_median64(st["phase"]), torch.log(_median64(st["amp"])), st["angles"], st["optics"],
                                case["iters"])}
    if kind == "steps":
        o = st["optics"]
        spec = _rytov(st["phase"].double(), st["logamp"].double())
        F, hits = _scatter(spec, st["angles"], case["V"], o)
        meas = F / hits.clamp(min=1.0) / o.dx
        return {"spec": spec, "hits": hits, "meas": meas,
                "ri": _loop64(torch.fft.ifftn(meas), meas, hits, case["iters"], o)}
    if kind == "fit":
        o, spec = st["optics"], st["spec"].to(torch.complex128)
        F, hits = _scatter(spec, st["angles"], case["V"], o)
        meas = F / hits.clamp(min=1.0) / o.dx
        return {"ri": _loop64(st["f0"].to(torch.complex128), meas, hits, case["iters"], o, case["step"])}
    out = []
    for c in st["cells"]:
        row, col = _search64(c["bg"][0])
        H = c["bg"].shape[-1]
        w, la = _retrieve64(c["holo"], c["bg"], row, col, abs(row - H // 2) // 3, c["V"])
        out.append(_volume64(_unwrap64(w, 0), la, c["angles"], c["optics"], c["iters"]))
    return {"ri": out, "crop": [None] * (2 * len(out))}
