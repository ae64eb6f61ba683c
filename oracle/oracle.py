"""FP64 CPU oracle for the standard gridder -- TEST INFRASTRUCTURE ONLY.

Imported only by tests/, by __graft_entry__.smoke() and by bench.py's
cpu_baseline leg, always as the checker and never as the thing measured or
shipped.  The product (astroviper_amd/) never imports this module.

The arithmetic lives in avgrid_oracle.c (a loop-by-loop C restatement of the
reference's numba kernels); this module adds the NumPy parts the reference
itself runs in NumPy (FFT + normalisation, argument preparation).  Reference
paths below are relative to src/astroviper/.
"""
from __future__ import annotations

import ctypes
import os
import subprocess

import numpy as np

_HERE = os.path.dirname(os.path.abspath(__file__))
_LIB_PATH = os.path.join(_HERE, "liboracle.so")
_lib = None

C_LIGHT = 299792458.0


def build(force: bool = False) -> str:
    """Compile liboracle.so with oracle/Makefile (gcc, no FMA contraction)."""
    if force or not os.path.exists(_LIB_PATH):
        subprocess.run(["make", "-s", "-C", _HERE, "-B" if force else "all"],
                       check=True)
    return _LIB_PATH


def lib():
    global _lib
    if _lib is None:
        if not os.path.exists(_LIB_PATH):
            build()
        L = ctypes.CDLL(_LIB_PATH)
        dp = ctypes.POINTER(ctypes.c_double)
        i64p = ctypes.POINTER(ctypes.c_int64)
        u8p = ctypes.POINTER(ctypes.c_uint8)
        I, I64, D = ctypes.c_int, ctypes.c_int64, ctypes.c_double
        L.ora_ps_function.argtypes = [dp, I64, dp, dp]
        L.ora_ps_kernel_1d.argtypes = [I, I, dp]
        L.ora_ps_taper.argtypes = [I, I, dp]
        L.ora_standard_grid.argtypes = [
            dp, I, dp, I, I, dp, I, dp, I, I, dp, I, i64p, i64p, I, dp, I, dp,
            I, I, I, I, D, D, I, I]
        L.ora_dgrid.argtypes = [dp, dp, u8p, I, I, I, I, dp, dp, dp, I, I, I,
                                I, dp, D, I, I, dp, i64p, i64p]
        L.ora_normalise.argtypes = [dp, dp, I64, I, I, dp, dp]
        L.ora_grid_geometry.argtypes = [D, D, D, D, D, I, I, I, I, i64p]
        L.ora_grid_geometry.restype = ctypes.c_int
        L.ora_degrid_geometry.argtypes = [dp, D, dp, dp, I, dp, i64p]
        L.ora_degrid_geometry.restype = None
        L.ora_grid_adjoint.argtypes = [dp, dp, u8p, I, I, I, I, dp, dp, dp, I, I, I, I, dp, D,
                                       I, I, dp, i64p, i64p]
        L.ora_grid_adjoint.restype = None
        L.ora_mosaic_grid.argtypes = [dp, dp, I, dp, I, dp, I, I, dp, I, i64p, i64p, I, i64p,
                                      i64p, i64p, dp, dp, I, I, I, I, I, I, I, D, D, i64p,
                                      I64, I, I]
        for f in (L.ora_ps_function, L.ora_ps_kernel_1d, L.ora_ps_taper,
                  L.ora_standard_grid, L.ora_dgrid, L.ora_normalise, L.ora_mosaic_grid):
            f.restype = None
        _lib = L
    return _lib


def _dp(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))


def _i64p(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_int64))


# --------------------------------------------------------------------------
# Kernel table and taper  (core/imaging/imaging_utils/gcf_prolate_spheroidal.py)
# --------------------------------------------------------------------------
def prolate_spheroidal_function(u):
    """gcf_prolate_spheroidal.py:102-158 -> (grdsf, (1-u^2)*grdsf)."""
    u = np.ascontiguousarray(np.asarray(u, dtype=np.float64))
    shp = u.shape
    uf = u.reshape(-1).copy()
    g = np.zeros_like(uf)
    k = np.zeros_like(uf)
    lib().ora_ps_function(_dp(uf), uf.size, _dp(g), _dp(k))
    return g.reshape(shp), k.reshape(shp)


def create_prolate_spheroidal_kernel_1D(oversampling, support):
    """gcf_prolate_spheroidal.py:87-99."""
    out = np.zeros(oversampling * (support // 2 + 1), dtype=np.float64)
    lib().ora_ps_kernel_1d(int(oversampling), int(support), _dp(out))
    return out


def coordinates(npixel):
    """gcf_prolate_spheroidal.py:161-163."""
    return (np.arange(npixel) - npixel // 2) / npixel


def create_prolate_spheroidal_kernel(oversampling, support, n_uv):
    """gcf_prolate_spheroidal.py:8-84: (4-D kernel, taper kernel_image)."""
    sc = support // 2
    oc = oversampling // 2
    sv = np.arange(support) - sc
    nrow = oversampling + 1 if oversampling % 2 == 0 else oversampling
    ovv = ((np.arange(nrow) - oc) / oversampling)[:, None]
    pts = (np.broadcast_to(sv, (nrow, support)) + ovv) / sc
    _, k1 = prolate_spheroidal_function(pts)
    kernel = np.zeros((nrow, nrow, support, support), dtype=np.double)
    for x in range(oversampling):
        for y in range(oversampling):
            kernel[x, y, :, :] = np.outer(k1[x, :], k1[y, :])
    taper = np.zeros((int(n_uv[0]), int(n_uv[1])), dtype=np.float64)
    lib().ora_ps_taper(int(n_uv[0]), int(n_uv[1]), _dp(taper))
    return kernel, taper


def grid_geometry(uvw_u, uvw_v, freq, cell, n_uv, support=7, oversampling=100):
    """standard_grid.py:296-352 for one sample -> (iu, iv, ou, ov) or None."""
    out = np.zeros(4, dtype=np.int64)
    ok = lib().ora_grid_geometry(float(uvw_u), float(uvw_v), float(freq), float(cell[0]),
                                 float(cell[1]), int(n_uv[0]), int(n_uv[1]), int(support),
                                 int(oversampling), _i64p(out))
    return tuple(int(x) for x in out) if ok else None


def degrid_geometry(uvw, freq, scale, offset, sampling):
    """sgrid_numba (standard_degrid.py:367-385) -> (pos[2], loc[2], off[2])."""
    u = np.ascontiguousarray(np.asarray(uvw, dtype=np.float64)[:3])
    sc = np.ascontiguousarray(np.asarray(scale, dtype=np.float64)[:2])
    of = np.ascontiguousarray(np.asarray(offset, dtype=np.float64)[:2])
    pos = np.zeros(2)
    lo = np.zeros(4, dtype=np.int64)
    lib().ora_degrid_geometry(_dp(u), float(freq), _dp(sc), _dp(of), int(sampling), _dp(pos),
                              _i64p(lo))
    return pos, lo[:2].copy(), lo[2:].copy()


# --------------------------------------------------------------------------
# Gridder  (core/imaging/imaging_utils/standard_grid.py)
# --------------------------------------------------------------------------
def standard_grid(vis, uvw, weight, freq_chan, n_uv, cell, support=7,
                  oversampling=100, chan_mode="continuum", do_psf=False,
                  grid=None, sum_weight=None, cgk_1D=None, complex_grid=True,
                  do_imaging_weight=False):
    """standard_grid_numpy_wrap (standard_grid.py:88-165) around the C
    restatement of standard_grid_jit (standard_grid.py:246-432).

    vis (nt, nb, nchan, nvispol) complex, uvw (nt, nb, 3), weight
    (nt, nb, nchan, npol).  Returns (grid, sum_weight), FP64.
    """
    weight = np.ascontiguousarray(weight, dtype=np.float64)
    uvw = np.ascontiguousarray(uvw, dtype=np.float64)
    freq_chan = np.ascontiguousarray(freq_chan, dtype=np.float64)
    nt, nb, nchan, npol = weight.shape
    if chan_mode == "cube":
        n_img_chan = nchan
        chan_map = np.arange(nchan, dtype=np.int64)
    else:
        n_img_chan = 1
        chan_map = np.zeros(nchan, dtype=np.int64)
    pol_map = np.arange(npol, dtype=np.int64)
    n_u, n_v = int(n_uv[0]), int(n_uv[1])
    if grid is None or (grid.size == 0 and sum_weight.size == 0):
        grid = np.zeros((n_img_chan, npol, n_u, n_v),
                        dtype=np.complex128 if complex_grid else np.float64)
        sum_weight = np.zeros((n_img_chan, npol), dtype=np.float64)
    if cgk_1D is None:
        cgk_1D = create_prolate_spheroidal_kernel_1D(oversampling, support)
    cgk_1D = np.ascontiguousarray(cgk_1D, dtype=np.float64)
    if do_psf:
        vis_c = np.zeros((1, 1, 1, 1), dtype=np.complex128)
        nvispol = 1
    else:
        vis_c = np.ascontiguousarray(vis, dtype=np.complex128)
        nvispol = vis_c.shape[3]
    assert grid.flags.c_contiguous and sum_weight.flags.c_contiguous
    lib().ora_standard_grid(
        _dp(grid.view(np.float64)), int(np.iscomplexobj(grid)),
        _dp(sum_weight), int(do_psf), int(do_imaging_weight),
        _dp(vis_c.view(np.float64)), nvispol, _dp(uvw), nt, nb,
        _dp(freq_chan), nchan, _i64p(chan_map), _i64p(pol_map), npol,
        _dp(weight), npol, _dp(cgk_1D), grid.shape[0], grid.shape[1], n_u, n_v,
        float(cell[0]), float(cell[1]), int(support), int(oversampling))
    return grid, sum_weight


def ifft_uv_to_lm(ary, axes):
    """core/imaging/ifft.py:5-18."""
    return np.fft.fftshift(np.fft.ifft2(np.fft.ifftshift(ary, axes=axes),
                                        axes=axes), axes=axes).real


def fft_lm_to_uv(ary, axes):
    """core/imaging/fft.py:5-18."""
    return np.fft.fftshift(np.fft.fft2(np.fft.ifftshift(ary, axes=axes),
                                       axes=axes), axes=axes)


def normalise(grid, sum_weight, support=7, oversampling=100):
    """standard_grid.py:693-708: per (chan, corr) plane
    real(fftshift(ifft2(ifftshift(grid)))) / corrTerm * nx * ny / sumwt."""
    nx, ny = grid.shape[-2:]
    _, corr = create_prolate_spheroidal_kernel(oversampling, support,
                                               np.array([nx, ny], dtype=int))
    out = np.zeros(grid.shape, dtype=np.float64)
    for ch in range(grid.shape[0]):
        for co in range(grid.shape[1]):
            out[ch, co] = (np.real(np.fft.fftshift(np.fft.ifft2(
                np.fft.ifftshift(grid[ch, co])))) / corr * nx * ny
                / sum_weight[ch, co])
    return out


def grid2image(vis, uvw, weight, flag, freq_chan, n_uv, cell, support=7,
               oversampling=100, chan_mode="continuum", do_psf=False):
    """grid2image_spheroid_ms4 (standard_grid.py:607-708) on plain arrays:
    weight is zeroed where flagged or where u/v is NaN (:664-668, on a copy
    here), the data are gridded, and the dirty image (or PSF) is formed.
    Returns (image, grid, sum_weight)."""
    weight = np.array(weight, dtype=np.float64, copy=True)
    if flag is not None:
        weight[np.asarray(flag, dtype=bool)] = 0.0
    nan_uvw = np.isnan(uvw[:, :, 0]) | np.isnan(uvw[:, :, 1])
    weight[nan_uvw] = 0.0
    grid, sw = standard_grid(vis, uvw, weight, freq_chan, n_uv, cell,
                             support=support, oversampling=oversampling,
                             chan_mode=chan_mode, do_psf=do_psf)
    img = normalise(grid, sw, support, oversampling)
    return img, grid, sw


# --------------------------------------------------------------------------
# Degridder  (core/imaging/imaging_utils/standard_degrid.py)
# --------------------------------------------------------------------------
def dgrid(uvw, values, flag, scale, offset, grid, freq, support, sampling,
          convFunc, chanmap, polmap, c=C_LIGHT):
    """dgrid_numba (standard_degrid.py:388-485), zero dphase, in place."""
    assert values.dtype == np.complex128 and values.flags.c_contiguous
    uvw = np.ascontiguousarray(uvw, dtype=np.float64)
    flag_u8 = np.ascontiguousarray(flag, dtype=np.uint8)
    grid_c = np.ascontiguousarray(grid, dtype=np.complex128)
    scale = np.ascontiguousarray(scale, dtype=np.float64)
    offset = np.ascontiguousarray(offset, dtype=np.float64)
    freq = np.ascontiguousarray(freq, dtype=np.float64)
    convFunc = np.ascontiguousarray(convFunc, dtype=np.float64)
    chanmap = np.ascontiguousarray(chanmap, dtype=np.int64)
    polmap = np.ascontiguousarray(polmap, dtype=np.int64)
    nt, nb, nvc, nvp = values.shape
    g = grid_c.shape
    lib().ora_dgrid(_dp(uvw), _dp(values.view(np.float64)),
                    flag_u8.ctypes.data_as(ctypes.POINTER(ctypes.c_uint8)),
                    nt, nb, nvc, nvp, _dp(scale), _dp(offset),
                    _dp(grid_c.view(np.float64)), g[0], g[1], g[2], g[3],
                    _dp(freq), float(c), int(support), int(sampling),
                    _dp(convFunc), _i64p(chanmap), _i64p(polmap))
    return values


def degrid(uvw, flag, freq, grid, cell, support=7, sampling=100,
           model=None):
    """degrid_spheroid_ms4 (standard_degrid.py:488-608) on plain arrays.
    NaN-uvw rows are flagged and their uvw set to 1e9 (:557-566, on copies
    here).  Returns the model visibilities, complex128."""
    uvw = np.array(uvw, dtype=np.float64, copy=True)
    flag = np.array(flag, dtype=bool, copy=True)
    nt, nb, nf, npl = flag.shape
    if model is None:
        model = np.zeros((nt, nb, nf, npl), dtype=np.complex128)
    nan_rows = np.isnan(uvw).any(axis=2)
    flag[nan_rows] = True
    uvw[nan_rows] = 1e9
    nx, ny = grid.shape[-2:]
    scale = np.array([-cell[0] * nx, -cell[1] * ny, 0.0], dtype=np.float64)
    offset = np.array([nx / 2, ny / 2, 0.0], dtype=np.float64)
    conv = create_prolate_spheroidal_kernel_1D(sampling, support)
    nchan, npol = grid.shape[0], grid.shape[1]
    chanmap = (np.arange(nf) / nf * nchan).astype(int)
    polmap = np.round(np.arange(npl) % npol).astype(int)
    return dgrid(uvw, model, flag, scale, offset, grid, freq, support,
                 sampling, conv, chanmap, polmap)


# --------------------------------------------------------------------------
# Measurement operator  A x = D F (x / t)  and its adjoint (no reference
# function; built from dgrid_numba, fft_lm_to_uv and the taper)
# --------------------------------------------------------------------------
def _degrid_setup(n_uv, cell, nf, nchan_g, npol_g, npl):
    nx, ny = n_uv
    scale = np.array([-cell[0] * nx, -cell[1] * ny, 0.0])
    offset = np.array([nx / 2, ny / 2, 0.0])
    chanmap = (np.arange(nf) / nf * nchan_g).astype(np.int64)
    polmap = (np.arange(npl) % npol_g).astype(np.int64)
    return scale, offset, chanmap, polmap


def grid_adjoint(uvw, values, flag, freq, n_uv, cell, nchan_g, npol_g, support=7,
                 sampling=100):
    """Transpose of degrid(): D^H y on a [nchan_g, npol_g, nx, ny] grid."""
    values = np.ascontiguousarray(values, dtype=np.complex128)
    nt, nb, nf, npl = values.shape
    scale, offset, chanmap, polmap = _degrid_setup(n_uv, cell, nf, nchan_g, npol_g, npl)
    grid = np.zeros((nchan_g, npol_g, int(n_uv[0]), int(n_uv[1])), dtype=np.complex128)
    conv = create_prolate_spheroidal_kernel_1D(sampling, support)
    fl = np.zeros(values.shape, np.uint8) if flag is None else np.ascontiguousarray(flag, np.uint8)
    u = np.ascontiguousarray(uvw, dtype=np.float64)
    f = np.ascontiguousarray(freq, dtype=np.float64)
    lib().ora_grid_adjoint(_dp(u), _dp(values.view(np.float64)),
                           fl.ctypes.data_as(ctypes.POINTER(ctypes.c_uint8)), nt, nb, nf, npl,
                           _dp(scale), _dp(offset), _dp(grid.view(np.float64)), nchan_g, npol_g,
                           grid.shape[2], grid.shape[3], _dp(f), C_LIGHT, int(support),
                           int(sampling), _dp(conv), _i64p(chanmap), _i64p(polmap))
    return grid


def measure(x, uvw, freq, cell, npol=1, support=7, sampling=100):
    """A x for an image x [nchan_g, npol_g, nx, ny]: degrid(fft_lm_to_uv(x / t))."""
    x = np.asarray(x)
    n_uv = x.shape[-2:]
    _, t = create_prolate_spheroidal_kernel(sampling, support, np.array(n_uv))
    g = fft_lm_to_uv(x / t, axes=[2, 3])
    nt, nb = uvw.shape[:2]
    flag = np.zeros((nt, nb, len(freq), npol), bool)
    return degrid(uvw, flag, freq, g, cell, support, sampling)


def measure_adjoint(y, uvw, freq, n_uv, cell, nchan_g=1, npol_g=1, support=7, sampling=100):
    """A^H y = fftshift(N^2 ifft2(ifftshift(D^H y))) / t."""
    g = grid_adjoint(uvw, y, None, freq, n_uv, cell, nchan_g, npol_g, support, sampling)
    _, t = create_prolate_spheroidal_kernel(sampling, support, np.array(n_uv))
    nn = n_uv[0] * n_uv[1]
    return np.fft.fftshift(np.fft.ifft2(np.fft.ifftshift(g, axes=[2, 3]), axes=[2, 3]),
                           axes=[2, 3]) * nn / t


# --------------------------------------------------------------------------
# Hogbom CLEAN  (core/imaging/deconvolvers/hogbom: src/hclean.cpp and the
# result dictionary of python/bindings.cpp:61-193)
# --------------------------------------------------------------------------
def _hogbom_lib(dtype):
    L = lib()
    sfx = "f32" if dtype == np.float32 else "f64"
    f = getattr(L, f"ora_hogbom_{sfx}")
    m = getattr(L, f"ora_maximg_{sfx}")
    if f.argtypes is None:
        T = ctypes.c_float if dtype == np.float32 else ctypes.c_double
        P = ctypes.c_void_p
        I = ctypes.c_int
        f.argtypes = [P, P, P, I, P, I, I, I, I, I, I, I, I, T, T, T, P]
        f.restype = I
        m.argtypes = [P, I, P, I, I, P, P]
        m.restype = None
    return f, m


def hogbom_maximg(image, mask=None):
    """maximg (hclean.cpp:51-81): (min, max) over the masked image."""
    img = np.ascontiguousarray(image)
    dt = np.float32 if img.dtype == np.float32 else np.float64
    img = img.astype(dt, copy=False)
    ny, nx = img.shape
    _, m = _hogbom_lib(dt)
    mk = None if mask is None or np.asarray(mask).size == 0 else \
        np.ascontiguousarray(mask, dtype=dt)
    lo, hi = np.zeros(1, dt), np.zeros(1, dt)
    m(img.ctypes.data, int(mk is not None), None if mk is None else mk.ctypes.data, nx, ny,
      lo.ctypes.data, hi.ctypes.data)
    return lo[0], hi[0]


def hogbom_clean(dirty_image, psf, mask=None, clean_box=(-1, -1, -1, -1), max_iter=100,
                 start_iter=0, gain=0.1, threshold=0.0, speedup=0.0):
    """clean (hclean.cpp:106-210 through bindings.cpp:61-193, no callbacks):
    the result dictionary of the reference's extension."""
    d = np.ascontiguousarray(dirty_image)
    # the overload the extension picks (bindings.cpp:243-301): float64 only
    # when every array given is float64, an empty mask included
    given = [d, np.asarray(psf)] + ([] if mask is None else [np.asarray(mask)])
    dt = np.float64 if all(a.dtype == np.float64 for a in given) else np.float32
    resid = d.astype(dt, copy=True)
    p = np.ascontiguousarray(psf, dtype=dt)
    ny, nx = resid.shape
    mk = None if mask is None or np.asarray(mask).size == 0 else \
        np.ascontiguousarray(mask, dtype=dt)
    xbeg, xend, ybeg, yend = 0, nx, 0, ny
    if len(clean_box) == 4:
        xbeg, xend, ybeg, yend = (int(v) for v in clean_box)
        xbeg = 0 if xbeg == -1 else xbeg
        xend = nx if xend == -1 else xend
        ybeg = 0 if ybeg == -1 else ybeg
        yend = ny if yend == -1 else yend
        xbeg = max(0, min(xbeg, nx - 1))
        xend = max(xbeg + 1, min(xend, nx))
        ybeg = max(0, min(ybeg, ny - 1))
        yend = max(ybeg + 1, min(yend, ny))
    model = np.zeros((ny, nx), dt)
    f, _ = _hogbom_lib(dt)
    it = f(model.ctypes.data, resid.ctypes.data, p.ctypes.data, int(mk is not None),
           None if mk is None else mk.ctypes.data, nx, ny, xbeg, xend, ybeg, yend,
           int(max_iter), int(start_iter), dt(gain), dt(threshold), dt(speedup), None)
    lo, hi = hogbom_maximg(resid, mk)
    final_peak = max(abs(lo), abs(hi))
    total = dt(0)
    for v in np.abs(model).ravel():  # the binding's sequential sum (bindings.cpp:175-178)
        total = dt(total + v)
    return {"model_image": model, "residual_image": resid, "iterations_performed": it,
            "final_peak": final_peak, "total_flux_cleaned": total,
            "converged": bool(final_peak <= dt(threshold))}


# --------------------------------------------------------------------------
# Imaging weights (core/imaging/imaging_weighting)
# --------------------------------------------------------------------------
def grid_imaging_weights(grid, sum_weight, uvw, data_weight, freq_chan, n_uv, cell):
    """grid_imaging_weights (grid_imaging_weights.py:7-100 ->
    grid_imaging_weights_jit :105-206) in place: grid (n_chan, 1, n_u, n_v)
    float64, sum_weight (n_chan, 1); data_weight (nt, nb, nchan, npol),
    polarisation 0 is gridded."""
    L = lib()
    f = L.ora_grid_imaging_weights
    if f.argtypes is None:
        P, I, D = ctypes.c_void_p, ctypes.c_int, ctypes.c_double
        f.argtypes = [P, P, P, I, I, P, I, P, I, I, I, D, D]
        f.restype = None
    assert grid.dtype == np.float64 and grid.flags.c_contiguous
    assert sum_weight.dtype == np.float64 and sum_weight.flags.c_contiguous
    u = np.ascontiguousarray(uvw, dtype=np.float64)
    w = np.ascontiguousarray(data_weight, dtype=np.float64)
    fr = np.ascontiguousarray(freq_chan, dtype=np.float64)
    nt, nb, nchan, npol = w.shape
    f(grid.ctypes.data, sum_weight.ctypes.data, u.ctypes.data, nt, nb, fr.ctypes.data, nchan,
      w.ctypes.data, npol, int(n_uv[0]), int(n_uv[1]), float(cell[0]), float(cell[1]))
    return grid, sum_weight


def degrid_imaging_weights(grid_imaging_weight, uvw, data_weight, briggs_factors, freq_chan,
                           n_uv, cell):
    """degrid_imaging_weights (grid_imaging_weights.py:209-271 ->
    degrid_imaging_weights_jit :274-443): per-sample imaging weights of
    shape data_weight (single polarisation, nt, nb, nchan, 1)."""
    L = lib()
    f = L.ora_degrid_imaging_weights
    if f.argtypes is None:
        P, I, D = ctypes.c_void_p, ctypes.c_int, ctypes.c_double
        f.argtypes = [P, P, P, P, I, I, P, I, P, I, I, D, D]
        f.restype = I
    w = np.ascontiguousarray(data_weight, dtype=np.float64)
    nt, nb, nchan, npol = w.shape
    assert npol == 1
    out = np.zeros(w.shape, dtype=np.float64)
    g = np.ascontiguousarray(grid_imaging_weight, dtype=np.float64)
    bf = np.ascontiguousarray(np.asarray(briggs_factors, dtype=np.float64).reshape(2, -1)[:, :nchan])
    u = np.ascontiguousarray(uvw, dtype=np.float64)
    fr = np.ascontiguousarray(freq_chan, dtype=np.float64)
    if f(out.ctypes.data, g.ctypes.data, bf.ctypes.data, u.ctypes.data, nt, nb, fr.ctypes.data,
         nchan, w.ctypes.data, int(n_uv[0]), int(n_uv[1]), float(cell[0]), float(cell[1])):
        raise ValueError("NaN in briggs_factors")
    return out


def calculate_briggs_params(grid_of_imaging_weights, sum_weight, imaging_weights_parms):
    """briggs_weighting.py:1-31 (NumPy, as the reference)."""
    if imaging_weights_parms["weighting"] == "briggs":
        robust = imaging_weights_parms["robust"]
        bf = np.ones((2,) + sum_weight.shape)
        sq = np.sum(grid_of_imaging_weights ** 2, axis=(2, 3))
        with np.errstate(invalid="ignore", divide="ignore"):
            bf[0, :, :] = (np.square(5.0 * 10.0 ** (-robust)) / (sq / sum_weight))[None, None, :, :]
    elif imaging_weights_parms["weighting"] == "briggs_abs":
        robust = imaging_weights_parms["robust"]
        bf = np.ones((2,) + sum_weight.shape)
        bf[0, :, :] = bf[0, :, :] * np.square(robust)
        bf[1, :, :] = bf[1, :, :] * 2.0 * np.square(imaging_weights_parms["briggs_abs_noise"])
    else:
        bf = np.zeros((2, 1, 1) + sum_weight.shape)
        bf[0, :, :] = np.ones((1, 1, 1) + sum_weight.shape)
    return bf


# --------------------------------------------------------------------------
# Mosaic / A-projection gridder  (core/imaging/imaging_utils/mosaic_grid.py)
# --------------------------------------------------------------------------
def mosaic_grid(grid, sum_weight, do_psf, vis_data, uvw, freq_chan, chan_map, pol_map,
                cf_baseline_map, cf_chan_map, cf_pol_map, imaging_weight, conv_kernel, n_uv,
                delta_lm, weight_support, oversampling, phase_gradient):
    """mosaic_grid_jit (mosaic_grid.py:306-486), accumulating into the
    complex `grid` [n_chan, n_pol, n_u, n_v] and `sum_weight` in place.
    conv_kernel [ncb, ncc, ncp, cu, cv] complex, phase_gradient [nfield, cu, cv];
    the product conv_kernel * phase_gradient[0] (mosaic_grid.py:359) is
    formed here with NumPy, as the reference does."""
    assert np.iscomplexobj(grid) and grid.flags.c_contiguous
    cfpg = np.ascontiguousarray(np.asarray(conv_kernel) * np.asarray(phase_gradient)[0, :, :],
                                dtype=np.complex128)
    ncb, ncc, ncp, cu_n, cv_n = cfpg.shape
    iw = np.ascontiguousarray(imaging_weight, dtype=np.float64)
    nt, nb, nchan, npol = iw.shape
    uvw = np.ascontiguousarray(uvw, dtype=np.float64)
    if do_psf:
        vis_c = np.zeros((1, 1, 1, 1), dtype=np.complex128)
        nvpol = 1
    else:
        vis_c = np.ascontiguousarray(vis_data, dtype=np.complex128)
        nvpol = vis_c.shape[3]
    ws = np.ascontiguousarray(weight_support, dtype=np.int64)
    i64 = lambda a: np.ascontiguousarray(a, dtype=np.int64)
    cm, pm, cbm, ccm, cpm = (i64(chan_map), i64(pol_map), i64(cf_baseline_map),
                             i64(cf_chan_map), i64(cf_pol_map))
    lib().ora_mosaic_grid(
        _dp(grid.view(np.float64)), _dp(sum_weight), int(do_psf), _dp(vis_c.view(np.float64)),
        nvpol, _dp(uvw), nt, nb, _dp(np.ascontiguousarray(freq_chan, dtype=np.float64)), nchan,
        _i64p(cm), _i64p(pm), npol, _i64p(cbm), _i64p(ccm), _i64p(cpm), _dp(iw),
        _dp(cfpg.view(np.float64)), ncc, ncp, cu_n, cv_n, grid.shape[1], int(n_uv[0]),
        int(n_uv[1]), float(delta_lm[0]), float(delta_lm[1]), _i64p(ws), int(np.max(ws)),
        int(oversampling[0]), int(oversampling[1]))
    return grid, sum_weight


# --------------------------------------------------------------------------
# Convolution functions of the mosaic gridder
# (core/imaging/make_gridding_convolution_function.py and
# core/imaging/imaging_utils/make_pb_symmetric.py), in NumPy/SciPy as the
# reference computes them.  The reference's make_phase_gradient projects the
# field direction with astropy's RA---SIN/DEC--SIN WCS, which is absent here;
# gcf_sin_offset restates that projection (zenithal SIN, native longitude of
# the pole 180 degrees, unit PC matrix).
# --------------------------------------------------------------------------
def gcf_aperture_patterns(freq_chan, pol, pb_params, grid_params, casa):
    """airy_disk_rorder (casa False) / casa_airy_disk_rorder (casa True),
    make_pb_symmetric.py:148-280: [n_ant_type, n_freq, n_pol, n0, n1]."""
    from scipy.special import jn
    cell = np.asarray(grid_params["cell_size"], dtype=np.float64)
    size = np.asarray(grid_params["image_size"])
    ctr = np.asarray(grid_params["image_center"])
    dishes = np.asarray(pb_params["list_dish_diameters"], dtype=np.float64)
    blocks = np.asarray(pb_params["list_blockage_diameters"], dtype=np.float64)
    ipower = pb_params["ipower"]
    kf = (2 * np.pi * np.asarray(freq_chan, dtype=np.float64)) / C_LIGHT
    x = np.arange(-ctr[0], size[0] - ctr[0]) * cell[0]
    y = np.arange(-ctr[1], size[1] - ctr[1]) * cell[1]
    xg, yg = np.meshgrid(x, y, indexing="ij")
    rad = np.sqrt(xg ** 2 + yg ** 2)
    out = np.zeros((len(blocks), len(kf), 1, size[0], size[1]))
    for a, (d, b) in enumerate(zip(dishes, blocks)):
        r = np.moveaxis(rad[:, :, None] * kf * (d / 2), 2, 0)
        r[:, ctr[0], ctr[1]] = 1.0
        if b == 0.0:
            v = 2.0 * jn(1, r) / r
        elif not casa:
            e = b / d
            v = (2.0 * jn(1, r) / r - 2.0 * e * jn(1, r * e) / r) / (1.0 - e ** 2)
        else:
            ar, lr = (d / b) ** 2, d / b
            v = (ar * 2.0 * jn(1, r) / r - 2.0 * jn(1, r * lr) / (r * lr)) / (ar - 1.0)
        out[a, :, 0] = v ** ipower
    out[:, :, 0, ctr[0], ctr[1]] = 1.0
    return np.tile(out, (1, 1, len(pol), 1, 1))


def gcf_baseline_patterns(pb_freq, pb_pol, pb_ant_pairs, casa, gcf_params, grid_params):
    """make_baseline_patterns (make_gridding_convolution_function.py:196-229)."""
    pgp = dict(grid_params)
    pgp["cell_size"] = np.asarray(grid_params["cell_size"]) * np.asarray(gcf_params["oversampling"])
    pgp["image_size"] = np.asarray(grid_params["image_size_padded"])
    pgp["image_center"] = pgp["image_size"] // 2
    pat = gcf_aperture_patterns(pb_freq, pb_pol, gcf_params, pgp, casa)
    n = pgp["image_size"]
    out = np.zeros((len(pb_ant_pairs), len(pb_freq), len(pb_pol), n[0], n[1]))
    for k, (i, j) in enumerate(pb_ant_pairs):
        out[k, :, 0] = pat[i, :, 0] * pat[j, :, 0]
    return out


def gcf_cf_baseline_map(unique_ant_indx, basline_ant, n_unique_ant):
    """create_cf_baseline_map (make_gridding_convolution_function.py:232-257)."""
    pairs = np.array([[i, j] for i in range(n_unique_ant) for j in range(i, n_unique_ant)],
                     dtype=int).reshape(-1, 2)
    u = np.asarray(unique_ant_indx)
    ba = np.asarray(basline_ant)
    t0, t1 = u[ba[:, 0]], u[ba[:, 1]]
    cbm = np.zeros(ba.shape[0], dtype=int)
    for k, (i, j) in enumerate(pairs):
        cbm[(t0 == i) & (t1 == j)] = k
    return cbm, pairs


def gcf_cf_chan_map(freq_chan, chan_tolerance_factor):
    """create_cf_chan_map (make_gridding_convolution_function.py:260-288)."""
    f = np.asarray(freq_chan, dtype=np.float64)
    n = len(f)
    tol = np.max(f) * chan_tolerance_factor
    npb = int(np.floor((np.max(f) - np.min(f)) / tol) + 0.5)
    npb = max(npb, 1)
    if npb >= n:
        return np.arange(n), f
    step = (np.max(f) - np.min(f)) / npb
    pb_freq = np.arange(npb) * step + np.min(f) + step / 2
    return np.array([int(np.argmin(np.abs(pb_freq - v))) for v in f]), pb_freq


def gcf_calc_conv_size(sub, imsize, support_cut_level, oversampling, max_support):
    """calc_conv_size (make_gridding_convolution_function.py:374-423)."""
    a = np.abs(sub)
    cut = support_cut_level * a.max()
    assert a.min() < cut
    out = []
    for ax in (0, 1):
        idx = [imsize[0] // 2, imsize[1] // 2]
        while sub[idx[0], idx[1]] > cut:
            idx[ax] += 1
            assert idx[ax] < imsize[ax]
        out.append((int(0.5 + (idx[ax] - imsize[ax] // 2) / oversampling[ax]) + 1) * 2 + 1)
    assert out[0] < max_support[0] and out[1] < max_support[1]
    s = max(out)
    return [s, s]


def gcf_resize_and_calc_support(ck, ckc, gcf_params, grid_params):
    """resize_and_calc_support (make_gridding_convolution_function.py:291-371)."""
    shp = ck.shape[:3]
    rcs = np.asarray(gcf_params["resize_conv_size"])
    ov = np.asarray(gcf_params["oversampling"])
    npad = np.asarray(grid_params["image_size_padded"])
    s0 = npad // 2 - rcs // 2
    e0 = s0 + rcs
    sup = np.zeros(shp + (2,), dtype=int)
    rk = np.zeros(shp + tuple(rcs))
    rkc = np.zeros(shp + tuple(rcs))
    for idx in np.ndindex(*shp):
        sup[idx] = gcf_calc_conv_size(ckc[idx], npad, gcf_params["support_cut_level"], ov,
                                      gcf_params["max_support"])
        emb = (sup[idx] + 1) * ov
        es = rcs // 2 - emb // 2
        ee = es + emb
        for src, dst in ((ck, rk), (ckc, rkc)):
            dst[idx] = src[idx][s0[0]:e0[0], s0[1]:e0[1]]
            dst[idx] = dst[idx] / np.real(np.sum(dst[idx][es[0]:ee[0], es[1]:ee[1]])
                                          / (ov[0] * ov[1]))
    return rk, rkc, sup


def gcf_sin_offset(field_dir, phase_center, cell):
    """Pixel offset of field_dir [n, 2] (RA, Dec radians) from the reference
    pixel of a RA---SIN/DEC--SIN image centred on phase_center with pixel
    steps cell (radians): (l / cell0, m / cell1) with l = cos d sin(a - a0),
    m = sin d cos d0 - cos d sin d0 cos(a - a0)."""
    fd = np.atleast_2d(np.asarray(field_dir, dtype=np.float64))
    a, d = fd[:, 0], fd[:, 1]
    a0, d0 = float(phase_center[0]), float(phase_center[1])
    l = np.cos(d) * np.sin(a - a0)
    m = np.sin(d) * np.cos(d0) - np.cos(d) * np.sin(d0) * np.cos(a - a0)
    return np.stack([l / cell[0], m / cell[1]], axis=1)


def gcf_phase_gradient(field_phase_dir, gcf_params, grid_params):
    """make_phase_gradient (make_gridding_convolution_function.py:426-485):
    [n_field, resize0, resize1] complex."""
    npad = np.asarray(grid_params["image_size_padded"])
    pd = gcf_sin_offset(field_phase_dir, np.asarray(gcf_params["phase_direction"]),
                        np.asarray(grid_params["cell_size"], dtype=np.float64))
    pix = -pd * 2 * np.pi / (npad * np.asarray(gcf_params["oversampling"]))
    size = np.asarray(gcf_params["resize_conv_size"])
    c = size // 2
    x = np.arange(-c[0], size[0] - c[0])
    y = np.arange(-c[1], size[1] - c[1])
    xg, yg = np.meshgrid(x, y, indexing="ij")
    return np.moveaxis(np.exp(1j * (xg[:, :, None] * pix[:, 0] + yg[:, :, None] * pix[:, 1])),
                       2, 0)
