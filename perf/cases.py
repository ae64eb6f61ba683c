"""Timed work of the framework: what its users call, over the sizes they call it with.

A case names a `kind` and its sizes.  The kinds:

grid      bin the uvw of one measurement set, grid its visibilities (or its
          weights, for the PSF) and degrid the grid back (GridPlan)
image     dirty image of a gridded cube (dirty_image)
cycle     predict, residual, grid and image of one major cycle on resident
          data (ResidentImager)
operator  chi-squared of the differentiable measurement operator and its
          gradient (MeasurementOperator)
clean     Hogbom CLEAN of every plane of a cube (ResidentImager.deconvolve)
weights   Briggs imaging weights of resident data (av_grid_imaging_weights,
          av_degrid_imaging_weights)
mosaic    bin and grid with baseline- and channel-dependent convolution
          functions (av_mosaic_grid)
planes    many image planes of uneven sample counts in one graph replay
          (BatchedGridder)
drop_in   the reference's entry points on host arrays: dirty image and model
          prediction of an MSv4 dataset
"""
import math

import numpy as np
import torch

from astroviper_amd import _lib
from astroviper_amd import device as D
from astroviper_amd.batch import BatchedGridder, PlaneSet
from astroviper_amd.major_cycle import ResidentImager
from astroviper_amd.measurement import MeasurementOperator
from astroviper_amd.mosaic_grid import _plan_shape
from astroviper_amd.msv4 import make_visibility_dataset
from astroviper_amd.standard_degrid import degrid_spheroid_ms4
from astroviper_amd.standard_grid import grid2image_spheroid_ms4

C_LIGHT = 299792458.0
DEV = "cuda"
SUPPORT, OVERSAMPLING = 7, 100


def _obs(n_ant, n_time, n_chan, n_pol, n_u, n_v, **more):
    return {"n_ant": n_ant, "n_time": n_time, "n_chan": n_chan, "n_pol": n_pol, "n_u": n_u,
            "n_v": n_v, **more}


def listed():
    return [
        # a short observation with the smallest array, in the reference's
        # precision: launches and latency
        {"name": "grid_snapshot_fp64", "kind": "grid", "mode": "cube", "precision": "fp64",
         "psf": False, "flags": False, "reach": 0.9, **_obs(27, 20, 4, 2, 128, 128)},
        # the benchmark's workload: a spectral-line cube, one plane per
        # channel and polarisation
        {"name": "grid_cube_fp32", "kind": "grid", "mode": "cube", "precision": "fp32",
         "psf": False, "flags": True, "reach": 1.8, **_obs(64, 1000, 64, 4, 2048, 2048)},
        # continuum imaging of two hands on a rectangular image that is not a
        # power of two: all channels on one plane
        {"name": "grid_continuum_fp32", "kind": "grid", "mode": "continuum",
         "precision": "fp32", "psf": False, "flags": True, "reach": 0.8,
         **_obs(64, 360, 48, 2, 1800, 1500)},
        # a cube in the reference's own precision
        {"name": "grid_cube_fp64", "kind": "grid", "mode": "cube", "precision": "fp64",
         "psf": False, "flags": True, "reach": 0.9, **_obs(64, 150, 16, 2, 1024, 1024)},
        # the image step of the cube: 32 of the benchmark's planes
        {"name": "image_cube", "kind": "image", "precision": "fp32", "n_chan": 8, "n_pol": 4,
         "n_u": 2048, "n_v": 2048},
        # a major cycle in the default precision
        {"name": "cycle_fp64", "kind": "cycle", "mode": "cube", "precision": "fp64",
         "reach": 0.9, **_obs(27, 200, 8, 2, 1024, 1024)},
        # one gradient of a sky model: 1024 x 1024 pixels, 1e7 samples
        {"name": "operator_fp32", "kind": "operator", "precision": "fp32", "reach": 0.45,
         **_obs(27, 7122, 4, 1, 1024, 1024)},
        # the minor cycle: 200 components per plane
        {"name": "clean_cube", "kind": "clean", "n_chan": 4, "n_pol": 2, "n_u": 1024,
         "n_v": 1024, "n_iter": 200},
        # Briggs weighting of the benchmark's array and image size
        {"name": "weights_briggs", "kind": "weights", "reach": 1.8,
         **_obs(64, 500, 32, 1, 2048, 2048)},
        # A-projection: 7 to 11 taps, 3 x 4 convolution functions
        {"name": "mosaic_cube_fp32", "kind": "mosaic", "precision": "fp32", "reach": 1.8,
         **_obs(64, 100, 32, 4, 2048, 2048)},
        # a batch of small images, one graph replay for all of them
        {"name": "planes_batch", "kind": "planes", "precision": "fp32", "n_planes": 96,
         "n_lo": 10000, "n_hi": 1000000, "n_u": 512, "n_v": 512},
        # the reference's calls on host arrays
        {"name": "drop_in_host", "kind": "drop_in", "mode": "cube", "reach": 0.9,
         **_obs(27, 100, 4, 2, 256, 256)},
    ]


# ------------------------------------------------------------------ draws --
def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """An image axis: most are even products of small primes, as imagers
    choose them, some are any number."""
    n = _log(rng, lo, hi)
    if rng.random() < 0.3:
        return n
    while True:
        m = n
        for p in (2, 3, 5):
            while m % p == 0:
                m //= p
        if m == 1 and n % 2 == 0:
            return n
        n += 1


def draw(rng):
    kind = rng.choice(["grid"] * 5 + ["image", "image", "cycle", "operator", "clean", "weights",
                                      "mosaic", "planes", "drop_in"])
    prec = rng.choice(["fp32", "fp64"])
    n_ant = rng.choice([27, 36, 64])
    nb = n_ant * (n_ant - 1) // 2
    reach = round(rng.uniform(0.5, 1.2), 2)
    mode = rng.choice(["cube", "continuum"])
    if kind == "image":
        n = _size(rng, 128, 2600)
        m = n if rng.random() < 0.7 else _size(rng, 128, 2600)
        planes = max(1, min(32, (1 << 26) // (n * m)))
        return {"kind": kind, "precision": prec, "n_chan": rng.randint(1, planes), "n_pol": 1,
                "n_u": n, "n_v": m}
    if kind == "clean":
        n = _size(rng, 128, 1600)
        return {"kind": kind, "n_chan": rng.randint(1, 4), "n_pol": rng.choice([1, 2]), "n_u": n,
                "n_v": n, "n_iter": _log(rng, 20, 300)}
    if kind == "planes":
        n = _size(rng, 128, 600)
        lo = _log(rng, 1000, 20000)
        return {"kind": kind, "precision": prec, "n_planes": rng.randint(6, 96), "n_lo": lo,
                "n_hi": lo * 50, "n_u": n, "n_v": n}
    n = _size(rng, 100, 2200)
    m = n if rng.random() < 0.6 else _size(rng, 100, 2200)
    n_pol = rng.choice([1, 2, 4])
    n_chan = _log(rng, 1, 64)
    n_chan = max(1, min(n_chan, (1 << 27) // (n * m * n_pol)))
    total = _log(rng, 2e4, 3e6 if kind in ("drop_in", "cycle") else 6e7)
    n_time = max(1, total // (nb * n_chan * n_pol))
    c = _obs(n_ant, n_time, n_chan, n_pol, n, m, kind=kind, reach=reach)
    if kind == "grid":
        c.update(mode=mode, precision=prec, psf=rng.random() < 0.2, flags=rng.random() < 0.7)
    elif kind == "operator":
        c.update(precision=prec, n_pol=1, n_time=max(1, min(n_time, 10_000_000 // (nb * n_chan))))
    elif kind == "weights":
        c.update(n_pol=1)
    elif kind == "mosaic":
        c.update(precision=prec, n_time=max(1, min(n_time, 20_000_000 // (nb * n_chan * n_pol))))
    elif kind == "cycle":
        c.update(mode=mode, precision=prec)
    elif kind == "drop_in":
        c.update(mode=mode)
    return c


# ----------------------------------------------------------------- inputs --
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 1000003 + 17)
    return g


def _types(case):
    if case.get("precision", "fp64") == "fp32":
        return torch.complex64, torch.float32
    return torch.complex128, torch.float64


def _rand(gen, *shape):
    return torch.rand(shape, generator=gen, device=DEV, dtype=torch.float64)


def _uvw(case, gen):
    """(uvw [time * baseline, 3] in metres, freq [n_chan], cell): antennas in
    a disc of 20 km, four hours of earth rotation at declination 30 degrees;
    the longest baseline at the highest frequency lies at `reach` of the
    grid's half width."""
    n_ant, n_time = case["n_ant"], case["n_time"]
    r = 20e3 * _rand(gen, n_ant).sqrt()
    th = 2 * math.pi * _rand(gen, n_ant)
    e, n = r * torch.cos(th), r * torch.sin(th)
    i, j = torch.triu_indices(n_ant, n_ant, offset=1, device=DEV)
    lat, dec = math.radians(34.0784), math.radians(30.0)
    x, y, z = -math.sin(lat) * n, e, math.cos(lat) * n
    lx, ly, lz = x[j] - x[i], y[j] - y[i], z[j] - z[i]
    h = torch.linspace(-2.0, 2.0, n_time, device=DEV, dtype=torch.float64)[:, None] * math.pi / 12
    sd, cd = math.sin(dec), math.cos(dec)
    uu = torch.sin(h) * lx + torch.cos(h) * ly
    vv = -sd * torch.cos(h) * lx + sd * torch.sin(h) * ly + cd * lz
    ww = cd * torch.cos(h) * lx - cd * torch.sin(h) * ly + sd * lz
    uvw = torch.stack([uu, vv, ww], dim=2).reshape(-1, 3).contiguous()
    freq = torch.linspace(1.0e9, 1.4e9, case["n_chan"], device=DEV, dtype=torch.float64)
    longest = float(torch.hypot(uvw[:, 0], uvw[:, 1]).max())
    cell = case["reach"] * C_LIGHT / (2 * float(freq[-1]) * longest)
    return uvw, freq, (-cell, cell)


def _visibilities(case, gen, uvw, freq, cell):
    """vis, weight, flag [rows, n_chan, n_pol]: three point sources and noise,
    weights in [0.5, 1.5], a tenth flagged."""
    cdt, rdt = _types(case)
    rows, nf, npol = uvw.shape[0], freq.numel(), case["n_pol"]
    field = abs(cell[0]) * min(case["n_u"], case["n_v"])
    lm = (_rand(gen, 3, 2) - 0.5) * 0.6 * field
    flux = (0.3 + _rand(gen, 3)).tolist()
    path = uvw[:, :2] @ lm.T
    vis = torch.empty((rows, nf, npol), dtype=cdt, device=DEV)
    step = max(1, (1 << 24) // max(1, rows))
    for a in range(0, nf, step):
        f = freq[a:a + step] * (-2 * math.pi / C_LIGHT)
        acc = 0
        for s, amp in enumerate(flux):
            ph = path[:, s:s + 1] * f
            acc = acc + torch.polar(torch.full_like(ph, amp), ph)
        noise = torch.randn((rows, f.numel(), npol, 2), generator=gen, device=DEV, dtype=rdt)
        vis[:, a:a + step] = acc[..., None].to(cdt) + torch.view_as_complex(noise) * 0.05
    weight = torch.empty((rows, nf, npol), dtype=rdt, device=DEV).uniform_(0.5, 1.5, generator=gen)
    flag = torch.empty((rows, nf, npol), dtype=torch.float32, device=DEV).uniform_(generator=gen)
    return vis, weight, flag < 0.1


def _image_channels(case):
    """(image channels, channel map [n_chan] int32)."""
    n = case["n_chan"]
    if case["mode"] == "cube":
        return n, torch.arange(n, dtype=torch.int32, device=DEV)
    return 1, torch.zeros(n, dtype=torch.int32, device=DEV)


def _sky(case, gen, planes, dtype):
    """[planes, n_u, n_v] images of Gaussian blobs."""
    n, m = case["n_u"], case["n_v"]
    y = torch.arange(n, device=DEV, dtype=torch.float64)[:, None]
    x = torch.arange(m, device=DEV, dtype=torch.float64)[None, :]
    out = torch.zeros((planes, n, m), dtype=torch.float64, device=DEV)
    for _ in range(12):
        cy, cx, s, a = _rand(gen, 4).tolist()
        s = 2 * (2.0 + 8.0 * s) ** 2
        spot = (torch.exp(-(y - (0.1 + 0.8 * cy) * n) ** 2 / s)
                * torch.exp(-(x - (0.1 + 0.8 * cx) * m) ** 2 / s))
        out += (0.1 + a) * _rand(gen, planes)[:, None, None] * spot
    return out.to(dtype)


def _host_dataset(case, gen):
    uvw, freq, cell = _uvw(case, gen)
    vis, weight, flag = _visibilities(case, gen, uvw, freq, cell)
    nt, nb = case["n_time"], uvw.shape[0] // case["n_time"]
    shape = (nt, nb) + tuple(vis.shape[1:])
    host = lambda t, s: np.ascontiguousarray(t.cpu().numpy().reshape(s))  # noqa: E731
    ms = make_visibility_dataset(host(vis, shape).astype(np.complex128), host(uvw, (nt, nb, 3)),
                                 host(weight, shape).astype(np.float64), host(flag, shape),
                                 freq.cpu().numpy())
    return ms, cell, uvw, freq, vis, weight, flag


def _psf_and_dirty(case, gen):
    """A PSF from the array's uv coverage and the dirty images of some point
    sources: psf [chan, 1, n, m], dirty [chan, pol, n, m], both float64."""
    n, m, nc, npol = case["n_u"], case["n_v"], case["n_chan"], case["n_pol"]
    obs = _obs(27, 60, nc, npol, n, m, reach=0.8)
    uvw, freq, cell = _uvw(obs, gen)
    psf = torch.empty((nc, 1, n, m), dtype=torch.float64, device=DEV)
    dirty = torch.empty((nc, npol, n, m), dtype=torch.float64, device=DEV)
    ax = (-2, -1)
    for c in range(nc):
        iu = (uvw[:, 0] * (freq[c] * cell[0] * n / C_LIGHT)).round().long()
        iv = (uvw[:, 1] * (freq[c] * cell[1] * m / C_LIGHT)).round().long()
        ok = (iu.abs() < n // 2) & (iv.abs() < m // 2)
        iu, iv = iu[ok], iv[ok]
        g = torch.zeros(n * m, dtype=torch.float64, device=DEV)
        for s in (1, -1):
            g += torch.bincount((s * iu) % n * m + (s * iv) % m, minlength=n * m)
        g = g.sqrt().reshape(n, m)
        beam = torch.fft.ifft2(g).real
        psf[c, 0] = torch.roll(beam / beam[0, 0], (n // 2, m // 2), ax)
        for p in range(npol):
            sky = torch.zeros((n, m), dtype=torch.float64, device=DEV)
            at = (_rand(gen, 12, 2) * 0.6 + 0.2) * torch.tensor([n, m], device=DEV)
            sky[at[:, 0].long(), at[:, 1].long()] = 0.05 + _rand(gen, 12)
            img = torch.fft.ifft2(torch.fft.fft2(sky) * g).real / beam[0, 0]
            noise = torch.randn((n, m), generator=gen, device=DEV, dtype=torch.float64)
            dirty[c, p] = img + 1e-3 * noise
    return psf, dirty


def _convolution_functions(gen):
    """weight_support [3, 4, 1, 2], functions times phase gradient
    [3, 4, 1, cu, cv] complex128; oversampling 8."""
    ws = 7 + 2 * torch.randint(0, 3, (3, 4, 1, 2), generator=gen, device=DEV, dtype=torch.int32)
    ws[0, 0, 0, 0] = 11
    k = 8 * (11 + 1) + 1
    x = (torch.arange(k, device=DEV, dtype=torch.float64) - k // 2) / k
    p = _rand(gen, 3, 4, 1, 3, 1, 1)
    a, b, ph = 4 + 4 * p[..., 0, :, :], 4 + 4 * p[..., 1, :, :], 6 * p[..., 2, :, :] - 3
    amp = torch.exp(-a * x[:, None] ** 2 - b * x[None, :] ** 2)
    ramp = torch.polar(torch.ones_like(amp), ph * (x[:, None] + 0.5 * x[None, :])
                       + 0.6 * (_rand(gen, k, k) - 0.5))
    return ws, amp * ramp


def _plane_sets(case, gen):
    """Plane sets of supports 5, 7 and 9 with log-uniform sample counts."""
    cdt, rdt = _types(case)
    n_pl, longest = case["n_planes"], 40e3
    cell = 0.95 * C_LIGHT / (2 * 1.4e9 * longest)
    # the same counts for every seed: they are the batch's shape
    spread = (torch.arange(n_pl, device=DEV, dtype=torch.float64) * 0.6180339887498949) % 1.0
    span = math.log(case["n_hi"] / case["n_lo"])
    counts = (case["n_lo"] * torch.exp(span * spread)).round().long()
    freqs = torch.linspace(1.0e9, 1.4e9, n_pl, device=DEV, dtype=torch.float64)
    sets = []
    for k, support in enumerate((5, 7, 9)):
        mine = torch.arange(k, n_pl, 3, device=DEV)
        cnt = counts[mine]
        plane = torch.repeat_interleave(
            torch.arange(mine.numel(), device=DEV, dtype=torch.int32), cnt)
        total = plane.numel()
        r = longest * _rand(gen, total)
        th = 2 * math.pi * _rand(gen, total)
        uvw = torch.stack([r * torch.cos(th), r * torch.sin(th), 0.1 * r], dim=1)
        vis = torch.randn((total, 1), generator=gen, device=DEV, dtype=cdt)
        weight = 0.5 + _rand(gen, total, 1).to(rdt)
        flag = (_rand(gen, total, 1) < 0.3).to(torch.uint8)
        sets.append(PlaneSet(support=support, uvw=uvw, plane=plane, freq=freqs[mine], vis=vis,
                             weight=weight, flag=flag))
    return sets, (-cell, cell)


# -------------------------------------------------------------- the cases --
def prepare(case, seed):
    gen = _gen(seed)
    kind = case["kind"]
    s = {"case": case}
    n_uv = (case["n_u"], case["n_v"])
    cdt, rdt = _types(case)
    if kind == "grid":
        s["uvw"], s["freq"], cell = _uvw(case, gen)
        vis, weight, flag = _visibilities(case, gen, s["uvw"], s["freq"], cell)
        flat = (-1, case["n_pol"])
        s["vis"], s["weight"] = vis.reshape(flat), weight.reshape(flat)
        s["flag"] = flag.reshape(flat) if case["flags"] else None
        n_img, s["map"] = _image_channels(case)
        rows = s["uvw"].shape[0]
        s["plan"] = D.GridPlan(rows, case["n_chan"], n_img, n_uv, cell, SUPPORT, OVERSAMPLING,
                               n_baseline=rows // case["n_time"])
    elif kind == "image":
        # uv data concentrated at short spacings, as a gridded cube has it
        shape = (case["n_chan"], case["n_pol"]) + n_uv
        r = [torch.linspace(-1, 1, n, device=DEV, dtype=rdt) for n in n_uv]
        fall = torch.exp(-4 * (r[0][:, None] ** 2 + r[1][None, :] ** 2))
        s["grid"] = torch.randn(shape, generator=gen, device=DEV, dtype=cdt)
        s["grid"] *= fall
        s["sumwt"] = 1e4 * (0.5 + _rand(gen, *shape[:2]))
    elif kind == "cycle":
        ms, cell = _host_dataset(case, gen)[:2]
        s["imager"] = ResidentImager(ms, n_uv, cell, SUPPORT, OVERSAMPLING, case["mode"],
                                     case["precision"])
        n_img = s["imager"].n_img_chan
        s["model"] = _sky(case, gen, n_img * case["n_pol"], torch.float64).reshape(
            (n_img, case["n_pol"]) + n_uv)
    elif kind == "operator":
        uvw, freq, cell = _uvw(case, gen)
        s["op"] = MeasurementOperator(uvw, freq, n_uv, cell, n_pol=1,
                                      chan_map=torch.zeros(freq.numel(), dtype=torch.int32,
                                                           device=DEV), dtype=cdt)
        s["data"] = torch.randn((s["op"].n_samples, 1), generator=gen, device=DEV, dtype=cdt)
        s["sky"] = _sky(case, gen, 1, rdt)[None].requires_grad_(True)
    elif kind == "clean":
        tiny = _obs(27, 1, 1, 1, case["n_u"], case["n_v"], reach=0.5)
        ms, cell = _host_dataset(tiny, gen)[:2]
        s["imager"] = ResidentImager(ms, n_uv, cell)
        s["psf"], s["dirty"] = _psf_and_dirty(case, gen)
    elif kind == "weights":
        s["uvw"], s["freq"], s["cell"] = _uvw(case, gen)
        w = 0.5 + _rand(gen, s["uvw"].shape[0], case["n_chan"])
        s["weight"] = torch.where(_rand(gen, *w.shape) < 0.1, math.nan, w)
    elif kind == "mosaic":
        s["uvw"], s["freq"], cell = _uvw(case, gen)
        vis, weight, flag = _visibilities(case, gen, s["uvw"], s["freq"], cell)
        s["vis"] = vis
        s["weight"] = torch.where(flag, torch.zeros_like(weight), weight)
        s["support"], cf = _convolution_functions(gen)
        s["cf"] = cf.to(cdt).contiguous()
        rows = s["uvw"].shape[0]
        nb = rows // case["n_time"]
        s["maps"] = [torch.arange(nb, dtype=torch.int32, device=DEV) % 3,
                     (torch.arange(case["n_chan"], device=DEV) * 4 // case["n_chan"]).int(),
                     torch.zeros(case["n_pol"], dtype=torch.int32, device=DEV)]
        support, tile = _plan_shape(11)
        s["plan"] = D.GridPlan(rows, case["n_chan"], case["n_chan"], n_uv, cell, support, 8,
                               tile=(tile, tile), n_baseline=nb)
    elif kind == "planes":
        sets, cell = _plane_sets(case, gen)
        s["gridder"] = BatchedGridder(sets, n_uv, cell)
        s["gridder"].capture()
    elif kind == "drop_in":
        s["ms"], cell = _host_dataset(case, gen)[:2]
        s["cell"] = np.array(cell)
        n_img = _image_channels(case)[0]
        s["shape"] = (n_img, case["n_pol"]) + n_uv
        m = _sky(case, gen, n_img * case["n_pol"], torch.float64).to(torch.complex128)
        s["model"] = torch.fft.fftshift(torch.fft.fft2(m), dim=(-2, -1)).reshape(
            s["shape"]).cpu().numpy()
    torch.cuda.synchronize()
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "grid":
        plan = s["plan"].set_uvw(s["uvw"], s["freq"], s["map"])
        grid, sumwt = plan.grid(s["vis"], s["weight"], s["flag"], psf=case["psf"])
        return {"grid": grid, "sumwt": sumwt, "model": plan.degrid(grid, s["flag"])}
    if kind == "image":
        return D.dirty_image(s["grid"], s["sumwt"], SUPPORT, OVERSAMPLING)
    if kind == "cycle":
        im = s["imager"]
        im.predict_model_visibilities(s["model"])
        im.compute_residual_visibilities()
        image = im.grid_visibilities("RESIDUAL")
        return {"model": im.model_vis, "residual": im.residual_vis, "image": image}
    if kind == "operator":
        s["sky"].grad = None
        y = s["op"].apply(s["sky"])
        (y - s["data"]).abs().pow(2).sum().backward()
        return {"visibilities": y.detach(), "gradient": s["sky"].grad}
    if kind == "clean":
        comps, resid, iters = s["imager"].deconvolve(s["dirty"], s["psf"], case["n_iter"],
                                                     gain=0.1, threshold=0.0)
        return {"components": comps, "residual": resid, "iterations": iters}
    if kind == "weights":
        return _run_weights(s, case)
    if kind == "mosaic":
        return _run_mosaic(s, case)
    if kind == "planes":
        g = s["gridder"]
        g.replay()
        return {"grids": list(g.grids), "sumwts": list(g.sumwts), "models": list(g.models)}
    image = np.zeros(s["shape"])
    grid2image_spheroid_ms4(s["ms"], image, s["cell"], SUPPORT, OVERSAMPLING,
                            chan_mode=case["mode"])
    degrid_spheroid_ms4(s["ms"], s["model"], s["cell"], SUPPORT, OVERSAMPLING)
    return {"image": image, "model": s["ms"]["VISIBILITY_MODEL"].data}


def _run_weights(s, case, robust=0.5):
    p, stream = D._ptr, D._stream()
    rows, nf, n, m = s["uvw"].shape[0], case["n_chan"], case["n_u"], case["n_v"]
    nb = rows // case["n_time"]
    grid = torch.zeros((nf, n, m), dtype=torch.float64, device=DEV)
    sw = torch.zeros(nf, dtype=torch.float64, device=DEV)
    _lib.call("av_grid_imaging_weights", p(s["uvw"]), rows, nb, p(s["freq"]), nf, p(s["weight"]),
              1, n, m, s["cell"][0], s["cell"][1], p(grid), p(sw), stream)
    square = torch.linalg.vector_norm(grid.reshape(nf, -1), dim=1) ** 2
    factors = torch.ones((2, nf), dtype=torch.float64, device=DEV)
    factors[0] = (5.0 * 10.0 ** -robust) ** 2 * sw / square
    out = torch.zeros((rows, nf), dtype=torch.float64, device=DEV)
    bad = torch.zeros(1, dtype=torch.int32, device=DEV)
    _lib.call("av_degrid_imaging_weights", p(grid), p(factors), p(s["uvw"]), rows, nb,
              p(s["freq"]), nf, p(s["weight"]), n, m, s["cell"][0], s["cell"][1], p(out), p(bad),
              stream)
    return {"density": grid, "sumwt": sw, "imaging_weight": out}


def _run_mosaic(s, case):
    p = D._ptr
    nf, npol = case["n_chan"], case["n_pol"]
    cdt, rdt = _types(case)
    plan = s["plan"].set_uvw(s["uvw"], s["freq"],
                             torch.arange(nf, dtype=torch.int32, device=DEV))
    grid = torch.zeros((nf, npol, case["n_u"], case["n_v"]), dtype=cdt, device=DEV)
    sw = torch.zeros((nf, npol), dtype=torch.float64, device=DEV)
    k = s["cf"].shape[-1]
    _lib.call("av_mosaic_grid", plan._h, p(s["vis"]), p(s["weight"]), npol,
              s["uvw"].shape[0] // case["n_time"], p(s["maps"][0]), p(s["maps"][1]),
              p(s["maps"][2]), p(s["cf"]), 3, 4, 1, k, k, p(s["support"]), 8, 8, p(grid), p(sw),
              _lib.AV_F32 if rdt == torch.float32 else _lib.AV_F64, 0, D._stream())
    return {"grid": grid, "sumwt": sw}


def work(case):
    """Inputs once, outputs once; two operations per tap and component."""
    kind = case["kind"]
    f = 4 if case.get("precision", "fp64") == "fp32" else 8
    n, m = case["n_u"], case["n_v"]
    cells = n * m
    log = 2.5 * (math.log2(n) + math.log2(m))
    taps = SUPPORT * SUPPORT
    if kind in ("image", "clean"):
        planes = case["n_chan"] * case["n_pol"]
        if kind == "image":
            return {"bytes": planes * cells * (2 * f + 8), "flops": planes * cells * log}
        return {"bytes": cells * 8 * (planes * 3 + case["n_chan"]),
                "flops": planes * cells * 2 * case["n_iter"]}
    if kind == "planes":
        lo, hi, npl = case["n_lo"], case["n_hi"], case["n_planes"]
        samples = npl * (hi - lo) / math.log(hi / lo)
        return {"bytes": samples * (28 + 5 * f + 1) + npl * cells * 2 * f,
                "flops": samples * 2 * 52 * 4}
    rows = case["n_time"] * case["n_ant"] * (case["n_ant"] - 1) // 2
    samples = rows * case["n_chan"]
    V = samples * case["n_pol"]
    planes = case["n_pol"] * (1 if case.get("mode") == "continuum" or kind == "operator"
                              else case["n_chan"])
    grid = planes * cells * 2 * f
    flops = V * taps * 4
    if kind == "grid":
        return {"bytes": rows * 24 + V * (5 * f + (1 if case["flags"] else 0)) + grid,
                "flops": 2 * flops}
    if kind == "cycle":
        return {"bytes": V * (7 * f + 1) + planes * cells * 16,
                "flops": 2 * flops + 2 * planes * cells * log}
    if kind == "operator":
        return {"bytes": V * 4 * f + 2 * cells * f, "flops": 2 * flops + 4 * cells * log}
    if kind == "weights":
        return {"bytes": rows * 24 + V * 16 + case["n_chan"] * cells * 8, "flops": V * 40}
    if kind == "mosaic":
        return {"bytes": rows * 24 + V * 3 * f + grid, "flops": V * 81 * 8}
    return {"bytes": rows * 24 + V * (16 + 8 + 1 + 16) + planes * cells * 24,
            "flops": 2 * flops + planes * cells * log}


# ---------------------------------------------------------- 64-bit values --
def _ps(u):
    """grdsf and (1 - u^2) grdsf of Schwab's rational approximation (m = 6,
    alpha = 1) on [0, 1]."""
    u = np.abs(np.asarray(u, dtype=np.float64))
    P = [[8.203343e-2, -3.644705e-1, 6.278660e-1, -5.335581e-1, 2.312756e-1],
         [4.028559e-3, -3.697768e-2, 1.021332e-1, -1.201436e-1, 6.412774e-2]]
    Q = [[1.0, 8.212018e-1, 2.078043e-1], [1.0, 9.599102e-1, 2.918724e-1]]
    part = (u >= 0.75).astype(int)
    d = u * u - np.where(part == 1, 1.0, 0.75 ** 2)
    top = sum(np.take([P[0][k], P[1][k]], part) * d ** k for k in range(5))
    bot = sum(np.take([Q[0][k], Q[1][k]], part) * d ** k for k in range(3))
    g = np.where(u <= 1.0, top / bot, 0.0)
    return g, (1 - u * u) * g


def _table(support):
    half = support // 2
    t = np.zeros(OVERSAMPLING * (half + 1))
    i = np.arange(OVERSAMPLING * half)
    t[:i.size] = _ps(i / (half * OVERSAMPLING))[1]
    return torch.from_numpy(t).to(DEV)


def _taper(n, m):
    t = [torch.from_numpy(_ps(2 * ((np.arange(k) - k // 2) / k))[0]).to(DEV) for k in (n, m)]
    return t[0][:, None] * t[1][None, :]


def _grid_place(u, v, f, cell, n, m, ov=OVERSAMPLING):
    """Centre cells and kernel offsets of the gridder's rounding."""
    at = []
    for x, c, k in ((u, cell[0], n), (v, cell[1], m)):
        pos = x * (-(f * c * float(k)) / C_LIGHT) + float(k // 2)
        ci = (pos + 0.5).trunc().clamp(-1e9, 1e9).long()
        at.append((ci, ((ci - pos) * ov + 0.5).floor().clamp(-1e9, 1e9).long()))
    return at


def _degrid_place(u, v, f, cell, n, m):
    """Centre cells and kernel offsets of the degridder's rounding."""
    at = []
    for x, c, k in ((u, cell[0], n), (v, cell[1], m)):
        pos = -c * float(k) * x * f / C_LIGHT + k / 2
        loc = pos.round().clamp(-1e9, 1e9)
        at.append((loc.long(), ((loc - pos) * OVERSAMPLING).round().clamp(-1e9, 1e9).long()))
    return at


def _inside(at, n, m, support):
    h = support // 2
    (iu, _), (iv, _) = at
    e = support - h - 1
    return (iu - h >= 0) & (iu + max(h, e) < n) & (iv - h >= 0) & (iv + max(h, e) < m)


def _taps(at, m, support, table):
    """(cell index, kernel weight) of every tap."""
    (iu, ou), (iv, ov) = at
    h = support // 2
    for i in range(-h, support - h):
        wu = table[(OVERSAMPLING * i + ou).abs()]
        for j in range(-h, support - h):
            yield (iu + i) * m + iv + j, wu * table[(OVERSAMPLING * j + ov).abs()]


def _scatter(acc, at, n, m, support, table, data, norm_first=False):
    """acc [n * m, 2 k] += kernel x data [rows, 2 k] (over the kernel sum if
    norm_first); returns the kernel sums."""
    norm = 0
    for _, w in _taps(at, m, support, table):
        norm = norm + w
    if norm_first:
        data = torch.where(norm[:, None] != 0, data / norm[:, None], 0.0)
    for cell, w in _taps(at, m, support, table):
        acc.index_add_(0, cell, w[:, None] * data)
    return norm


def _gather(plane, at, m, support, table):
    """Kernel-weighted means of plane [n * m, 2 k]."""
    norm, out = 0, 0
    for cell, w in _taps(at, m, support, table):
        out = out + w[:, None] * plane[cell]
        norm = norm + w
    return torch.where(norm[:, None] != 0, out / norm[:, None], 0.0)


def _flat(z):
    """[rows, pol] complex as [rows, 2 pol] float64."""
    return torch.view_as_real(z.to(torch.complex128)).reshape(z.shape[0], -1)


def _exact_grid(case, uvw, freq, cell, vis, weight, flag, chan_map, n_img, psf=False):
    n, m, npol = case["n_u"], case["n_v"], case["n_pol"]
    table = _table(SUPPORT)
    acc = torch.zeros((n_img, n * m, 2 * npol), dtype=torch.float64, device=DEV)
    sumwt = torch.zeros((n_img, npol), dtype=torch.float64, device=DEV)
    for c in range(freq.numel()):
        at = _grid_place(uvw[:, 0], uvw[:, 1], freq[c], cell, n, m)
        ok = torch.nonzero(_inside(at, n, m, SUPPORT))[:, 0]
        at = [(a[ok], b[ok]) for a, b in at]
        w = weight[ok, c].double()
        if flag is not None:
            w = torch.where(flag[ok, c], 0.0, w)
        d = w.to(torch.complex128) if psf else vis[ok, c].to(torch.complex128) * w
        norm = _scatter(acc[chan_map[c]], at, n, m, SUPPORT, table, _flat(d))
        sumwt[chan_map[c]] += (torch.where(d != 0, w, 0.0) * norm[:, None]).sum(0)
    grid = torch.view_as_complex(acc.reshape(n_img, n, m, npol, 2))
    return grid.permute(0, 3, 1, 2).contiguous(), sumwt


def _exact_degrid(case, uvw, freq, cell, grid, flag, chan_map):
    n, m, npol = case["n_u"], case["n_v"], case["n_pol"]
    table = _table(SUPPORT)
    out = torch.zeros((uvw.shape[0], freq.numel(), npol), dtype=torch.complex128, device=DEV)
    for c in range(freq.numel()):
        at = _degrid_place(uvw[:, 0], uvw[:, 1], freq[c], cell, n, m)
        # the reference bounds u by the last axis too
        ok = torch.nonzero(_inside(at, min(n, m), min(n, m), SUPPORT) if n != m
                           else _inside(at, n, m, SUPPORT))[:, 0]
        at = [(a[ok], b[ok]) for a, b in at]
        plane = torch.view_as_real(grid[chan_map[c]].to(torch.complex128)).permute(
            1, 2, 0, 3).reshape(n * m, 2 * npol)
        got = _gather(plane, at, m, SUPPORT, table).reshape(-1, npol, 2)
        out[ok, c] = torch.view_as_complex(got.contiguous())
    if flag is not None:
        out[flag] = 0
    return out


def _exact_image(grid, sumwt):
    n, m = grid.shape[-2:]
    taper, ax = _taper(n, m), (-2, -1)
    out = torch.empty(grid.shape, dtype=torch.float64, device=DEV)
    for c in range(grid.shape[0]):
        g = grid[c].to(torch.complex128)
        img = torch.fft.fftshift(torch.fft.ifft2(torch.fft.ifftshift(g, dim=ax)), dim=ax).real
        out[c] = img / taper * n * m / sumwt[c][:, None, None]
    return out


def _to_uv(model):
    ax = (-2, -1)
    m = model.to(torch.complex128)
    return torch.fft.fftshift(torch.fft.fft2(torch.fft.ifftshift(m, dim=ax)), dim=ax)


def _exact_clean(case, psf, dirty):
    n, m = case["n_u"], case["n_v"]
    comps, resid = torch.zeros_like(dirty), torch.empty_like(dirty)
    iters = np.full(dirty.shape[:2], case["n_iter"], dtype=np.int64)
    gain = float(np.float32(0.1))
    for c in range(dirty.shape[0]):
        p = psf[c, 0].float().double()
        for q in range(dirty.shape[1]):
            r = dirty[c, q].float().double()
            for _ in range(case["n_iter"]):
                k = int(r.abs().argmax())
                y, x = divmod(k, m)
                pv = gain * float(r[y, x])
                comps[c, q, y, x] += pv
                y1, x1 = max(0, y - n // 2), max(0, x - m // 2)
                y2, x2 = min(n - 1, y + n // 2 - 1), min(m - 1, x + m // 2 - 1)
                oy, ox = n // 2 - y, m // 2 - x
                r[y1:y2 + 1, x1:x2 + 1] -= pv * p[y1 + oy:y2 + oy + 1, x1 + ox:x2 + ox + 1]
            resid[c, q] = r
    return {"components": comps, "residual": resid, "iterations": iters}


def _exact_weights(case, gen, robust=0.5):
    n, m, nf = case["n_u"], case["n_v"], case["n_chan"]
    uvw, freq, cell = _uvw(case, gen)
    w = 0.5 + _rand(gen, uvw.shape[0], nf)
    w = torch.where(_rand(gen, *w.shape) < 0.1, math.nan, w)
    grid = torch.zeros((nf, n * m), dtype=torch.float64, device=DEV)
    sw = torch.zeros(nf, dtype=torch.float64, device=DEV)
    out = torch.zeros_like(w)
    for c in range(nf):
        at, co = [], []
        for x, k, d in ((uvw[:, 0], n, cell[0]), (uvw[:, 1], m, cell[1])):
            u = x * (-(freq[c] * d * float(k)) / C_LIGHT)
            at.append((u + float(k // 2) + 0.5).trunc().long())
            co.append((-u + float(k // 2) + 0.5).trunc().long())
        ok = (at[0] >= 0) & (at[0] < n) & (at[1] >= 0) & (at[1] < m)
        use = ok & ~w[:, c].isnan()
        con = use & (co[0] >= 0) & (co[0] < n) & (co[1] >= 0) & (co[1] < m)
        pix = at[0] * m + at[1]
        grid[c].index_add_(0, pix[use], w[use, c])
        grid[c].index_add_(0, (co[0] * m + co[1])[con], w[con, c])
        sw[c] = 2 * w[use, c].sum()
        a = (5.0 * 10.0 ** -robust) ** 2 * sw[c] / (grid[c] ** 2).sum()
        g = grid[c][pix[ok]]
        wo = w[ok, c]
        out[ok, c] = torch.where(wo.isnan() | (wo == 0) | (g == 0), wo, wo / (a * g + 1.0))
    return {"density": grid.reshape(nf, n, m), "sumwt": sw, "imaging_weight": out}


def _exact_mosaic(case, s, cell):
    n, m, nf, npol = case["n_u"], case["n_v"], case["n_chan"], case["n_pol"]
    ws, cf = s["support"].cpu().numpy(), s["cf"].to(torch.complex128)
    k, top = cf.shape[-1], int(ws.max())
    acc = torch.zeros((nf, n * m, 2 * npol), dtype=torch.float64, device=DEV)
    sumwt = torch.zeros((nf, npol), dtype=torch.float64, device=DEV)
    bmap = s["maps"][0].repeat(case["n_time"])
    for c in range(nf):
        fc = int(s["maps"][1][c])
        (iu, ou), (iv, ov) = _grid_place(s["uvw"][:, 0], s["uvw"][:, 1], s["freq"][c], cell, n, m,
                                         8)
        ok = (iu - top >= 0) & (iu + top < n) & (iv - top >= 0) & (iv + top < m)
        for b in range(3):
            r = torch.nonzero(ok & (bmap == b))[:, 0]
            su, sv = (int(x) for x in ws[b, fc, 0])
            w = s["weight"][r, c].double()
            d = s["vis"][r, c].to(torch.complex128) * w
            norm = 0
            for i in range(-(su // 2), su - su // 2):
                for j in range(-(sv // 2), sv - sv // 2):
                    f = cf[b, fc, 0].reshape(-1)[(8 * i + ou[r] + k // 2) * k
                                                 + 8 * j + ov[r] + k // 2]
                    norm = norm + f
                    acc[c].index_add_(0, (iu[r] + i) * m + iv[r] + j, _flat(d * f[:, None]))
            sumwt[c] += (torch.where(d != 0, w, 0.0) * (norm * norm).real[:, None]).sum(0)
    grid = torch.view_as_complex(acc.reshape(nf, n, m, npol, 2))
    return {"grid": grid.permute(0, 3, 1, 2).contiguous(), "sumwt": sumwt}


def _exact_planes(case, gen):
    n, m = case["n_u"], case["n_v"]
    sets, cell = _plane_sets(case, gen)
    out = []
    for ps in sets:
        table, f = _table(ps.support), ps.freq[ps.plane.long()]
        off = ps.plane.long() * (n * m)
        fl = ps.flag[:, 0].bool()
        at = _grid_place(ps.uvw[:, 0], ps.uvw[:, 1], f, cell, n, m)
        ok = torch.nonzero(_inside(at, n, m, ps.support) & ~fl)[:, 0]
        at = [(a[ok], b[ok]) for a, b in at]
        w = ps.weight[ok].double()
        acc = torch.zeros((ps.n_planes * n * m, 2), dtype=torch.float64, device=DEV)
        data, norm = _flat(ps.vis[ok].to(torch.complex128) * w), 0
        for cell_i, k in _taps(at, m, ps.support, table):
            acc.index_add_(0, cell_i + off[ok], k[:, None] * data)
            norm = norm + k
        sw = torch.zeros(ps.n_planes, dtype=torch.float64, device=DEV).index_add_(
            0, ps.plane[ok].long(), w[:, 0] * norm)
        # the model is degridded from the grid as stored
        at = _degrid_place(ps.uvw[:, 0], ps.uvw[:, 1], f, cell, n, m)
        ok = torch.nonzero(_inside(at, n, m, ps.support) & ~fl)[:, 0]
        at = [(a[ok], b[ok]) for a, b in at]
        got, norm = 0, 0
        for cell_i, k in _taps(at, m, ps.support, table):
            got = got + k[:, None] * acc[cell_i + off[ok]]
            norm = norm + k
        model = torch.zeros((ps.n_samples, 1), dtype=torch.complex128, device=DEV)
        model[ok, 0] = torch.view_as_complex(got / norm[:, None])
        out.append((ps, torch.view_as_complex(acc.reshape(ps.n_planes, 1, n, m, 2)), sw[:, None],
                    model))
    out.sort(key=lambda t: -t[0].n_samples * t[0].support ** 2)
    return {"grids": [t[1] for t in out], "sumwts": [t[2] for t in out],
            "models": [t[3] for t in out]}


def exact(case, seed):
    gen = _gen(seed)
    kind = case["kind"]
    rows = (case["n_time"] * case["n_ant"] * (case["n_ant"] - 1) // 2 if "n_ant" in case else 0)
    if rows and rows * case["n_chan"] * case["n_pol"] > 600_000_000:
        return None
    if kind == "image":
        s = prepare(case, seed)
        return _exact_image(s["grid"], s["sumwt"])
    if kind == "clean":
        tiny = _obs(27, 1, 1, 1, case["n_u"], case["n_v"], reach=0.5)
        _host_dataset(tiny, gen)
        return _exact_clean(case, *_psf_and_dirty(case, gen))
    if kind == "weights":
        return _exact_weights(case, gen)
    if kind == "planes":
        return _exact_planes(case, gen)
    if kind == "mosaic":
        s = prepare(case, seed)
        return _exact_mosaic(case, s, s["plan"].cell)
    uvw, freq, cell = _uvw(case, gen)
    if kind == "operator":
        cdt, rdt = _types(case)
        data = torch.randn((rows * freq.numel(), 1), generator=gen, device=DEV, dtype=cdt)
        sky = _sky(case, gen, 1, rdt)[None].double()
        n, m = case["n_u"], case["n_v"]
        taper = _taper(n, m)
        zero = [0] * freq.numel()
        y = _exact_degrid(case, uvw, freq, cell, _to_uv(sky / taper), None, zero)
        r = 2 * (y.reshape(-1, 1) - data.to(torch.complex128)).reshape(rows, -1, 1)
        acc = torch.zeros((n * m, 2), dtype=torch.float64, device=DEV)
        for c in range(freq.numel()):
            at = _degrid_place(uvw[:, 0], uvw[:, 1], freq[c], cell, n, m)
            ok = torch.nonzero(_inside(at, min(n, m), min(n, m), SUPPORT) if n != m
                               else _inside(at, n, m, SUPPORT))[:, 0]
            at = [(a[ok], b[ok]) for a, b in at]
            _scatter(acc, at, n, m, SUPPORT, _table(SUPPORT), _flat(r[ok, c]), norm_first=True)
        g = torch.fft.ifftshift(torch.view_as_complex(acc.reshape(n, m, 2)))
        grad = torch.fft.fftshift(torch.fft.ifft2(g)).real * (n * m) / taper
        return {"visibilities": y.reshape(-1, 1), "gradient": grad[None, None]}
    vis, weight, flag = _visibilities(case, gen, uvw, freq, cell)
    n_img, chan_map = _image_channels(case)
    cmap = chan_map.tolist()
    if kind == "grid":
        flag = flag if case["flags"] else None
        grid, sumwt = _exact_grid(case, uvw, freq, cell, vis, weight, flag, cmap, n_img,
                                  case["psf"])
        model = _exact_degrid(case, uvw, freq, cell, grid, flag, cmap)
        return {"grid": grid, "sumwt": sumwt, "model": model.reshape(-1, case["n_pol"])}
    n_uv = (case["n_u"], case["n_v"])
    sky = _sky(case, gen, n_img * case["n_pol"], torch.float64).reshape(
        (n_img, case["n_pol"]) + n_uv)
    if kind == "cycle":
        model = _exact_degrid(case, uvw, freq, cell, _to_uv(sky), flag, cmap)
        resid = vis.to(torch.complex128) - model
        image = _exact_image(*_exact_grid(case, uvw, freq, cell, resid, weight, flag, cmap,
                                          n_img))
        flat = (-1, case["n_pol"])
        return {"model": model.reshape(flat), "residual": resid.reshape(flat), "image": image}
    image = _exact_image(*_exact_grid(case, uvw, freq, cell, vis, weight, flag, cmap, n_img))
    uv = torch.fft.fftshift(torch.fft.fft2(sky.to(torch.complex128)), dim=(-2, -1))
    model = _exact_degrid(case, uvw, freq, cell, uv, flag, cmap)
    nt = case["n_time"]
    return {"image": image, "model": model.reshape((nt, -1) + tuple(model.shape[1:]))}
