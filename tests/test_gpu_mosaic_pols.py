"""The mosaic gridder where polarisations share a convolution function (the
tile's rows go to the wavefronts) and where they do not (its polarisations
do), against the oracle: 1, 2 and 4 polarisations, a convolution function
whose sides are no multiple of the oversampling (so the last tap of some
phases is past it) or narrower than it, tiles cut by the grid's edge, and a
polarisation with no data where the function is not finite."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

C = 299792458.0


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("pol_maps,side", [([0], 47), ([0, 0], 47), ([1, 0], 5),
                                           ([1, 1, 1, 1], 47), ([1, 1, 1, 1], 5),
                                           ([0, 1, 1, 0], 47)])
def test_mosaic_polarisation_split(gpu, oracle, pol_maps, side, prec):
    from astroviper_amd import synth
    from astroviper_amd.mosaic_grid import mosaic_grid_jit
    npol, n_uv, ov = len(pol_maps), (131, 90), (6, 8)
    arr = synth.ArrayConfig(seed=3, n_ant=12, n_time=15, n_chan=2, n_pol=npol)
    obs = synth.make_observation(arr, synth.SkyConfig())
    vis, w, _ = synth.host_visibilities(obs, synth.SkyConfig(), flag_frac=0.0,
                                        weight_range=(0.5, 1.5))
    nt, nb, nchan, _ = w.shape
    maxuv = np.max(np.hypot(obs.uvw[..., 0], obs.uvw[..., 1]))
    c = 0.35 * C / obs.freq[-1] / maxuv
    rng = np.random.default_rng(side)
    cf = (rng.uniform(0.5, 1.5, size=(3, 2, 2, side, side + 1))
          + 0.2j * rng.normal(size=(3, 2, 2, side, side + 1)))
    cfbm, cfcm = np.arange(nb) % 3, np.array([1, 0])
    w[rng.random(w.shape) < 0.2] = 0.0
    if npol > 1:
        cf[2] = np.nan
        w[:, cfbm == 2, :, npol - 1] = 0.0
    if prec == 32:
        vis = vis.astype(np.complex64).astype(np.complex128)
        w = w.astype(np.float32).astype(np.float64)
        cf = cf.astype(np.complex64).astype(np.complex128)
    ws = rng.integers(3, 8, size=(3, 2, 2, 2))
    args = (obs.uvw, obs.freq, np.arange(nchan), np.arange(npol), cfbm, cfcm,
            np.array(pol_maps), w, cf, np.array(n_uv), (-c, c * n_uv[0] / n_uv[1]), ws,
            np.array(ov), np.ones((1,) + cf.shape[-2:], dtype=np.complex128))
    gref = np.zeros((nchan, npol) + n_uv, dtype=np.complex128)
    sref = np.zeros((nchan, npol))
    oracle.mosaic_grid(gref, sref, False, vis, *args)
    last = gref[:, -1]
    assert np.isfinite(last).all() and np.count_nonzero(last) > 500
    g = np.zeros(gref.shape, dtype=np.complex64 if prec == 32 else np.complex128)
    s = np.zeros_like(sref)
    mosaic_grid_jit(g, s, False, vis, *args)
    # each cell sums a few hundred products, each rounded once
    tol = 1e-5 if prec == 32 else 1e-12
    np.testing.assert_allclose(g, gref, rtol=0, atol=tol * np.nanmax(np.abs(gref)))
    np.testing.assert_allclose(s, sref, rtol=1e-6 if prec == 32 else 1e-12)


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("pol_maps,side,n_time", [
    ([0], 47, 373),        # 49,236 samples: the fewest whose kernel values are copied by phase
    ([0], 47, 372),        # one time fewer: read in the caller's order
    ([1, 1], 47, 400), ([1, 0], 5, 400), ([0, 1, 1, 0], 47, 400),
])
def test_mosaic_kernel_values_by_phase(gpu, oracle, pol_maps, side, n_time, prec):
    """Enough samples for kernel values by phase.  A cell sums some ten thousand
    products in FP32, each rounded to 2^-24 of a partial sum: about 1e-5 of the
    largest, 1e-4 at most."""
    from astroviper_amd import synth
    from astroviper_amd.mosaic_grid import mosaic_grid_jit
    npol, n_uv, ov = len(pol_maps), (131, 90), (6, 8)
    arr = synth.ArrayConfig(seed=5, n_ant=12, n_time=n_time, n_chan=2, n_pol=npol)
    obs = synth.make_observation(arr, synth.SkyConfig())
    nt, nb, nchan = n_time, 66, 2
    rng = np.random.default_rng(side + npol)
    shape = (nt, nb, nchan, npol)
    vis = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    w = rng.uniform(0.5, 1.5, shape)
    w[rng.random(shape) < 0.2] = 0.0
    maxuv = np.max(np.hypot(obs.uvw[..., 0], obs.uvw[..., 1]))
    c = 0.35 * C / obs.freq[-1] / maxuv
    cf = (rng.uniform(0.5, 1.5, size=(3, 2, 2, side, side + 1))
          + 0.2j * rng.normal(size=(3, 2, 2, side, side + 1)))
    if prec == 32:
        vis = vis.astype(np.complex64).astype(np.complex128)
        w = w.astype(np.float32).astype(np.float64)
        cf = cf.astype(np.complex64).astype(np.complex128)
    ws = rng.integers(3, 8, size=(3, 2, 2, 2))
    args = (obs.uvw, obs.freq, np.arange(nchan), np.arange(npol), np.arange(nb) % 3,
            np.array([1, 0]), np.array(pol_maps), w, cf, np.array(n_uv),
            (-c, c * n_uv[0] / n_uv[1]), ws, np.array(ov),
            np.ones((1,) + cf.shape[-2:], dtype=np.complex128))
    gref = np.zeros((nchan, npol) + n_uv, dtype=np.complex128)
    sref = np.zeros((nchan, npol))
    oracle.mosaic_grid(gref, sref, False, vis, *args)
    assert np.count_nonzero(gref[:, -1]) > 500
    g = np.zeros(gref.shape, dtype=np.complex64 if prec == 32 else np.complex128)
    s = np.zeros_like(sref)
    mosaic_grid_jit(g, s, False, vis, *args)
    tol = 1e-4 if prec == 32 else 1e-12
    np.testing.assert_allclose(g, gref, rtol=0, atol=tol * np.max(np.abs(gref)))
    np.testing.assert_allclose(s, sref, rtol=1e-6 if prec == 32 else 1e-12)
