"""CLEAN of many planes in one call (clean_planes_device) where its layout
changes: one or several workgroups, columns and rows that do not fill a
wavefront's tile, more planes than run side by side, planes too large for the
registers, PSFs shared by planes; bit-identical with the oracle's CLEAN of each
plane, as the single-plane call is."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


def _planes(n, ny, nx, n_psf, dt, seed):
    rng = np.random.default_rng(seed)
    yy, xx = np.mgrid[0:ny, 0:nx]
    psf = np.stack([np.exp(-((xx - nx // 2) ** 2 + (yy - ny // 2) ** 2) / (4.0 + k))
                    for k in range(n_psf)]).astype(dt)
    return rng.standard_normal((n, ny, nx)).astype(dt), psf


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("n,ny,nx,per_psf,iters", [
    (1, 1, 1, 1, 3),          # one pixel
    (3, 5, 64, 1, 20),        # one wavefront, fewer rows than a tile
    (5, 9, 65, 2, 20),        # a second column tile of one lane
    (4, 130, 127, 4, 30),     # odd axes
    (2, 600, 200, 1, 30),     # several workgroups per plane
    (300, 64, 64, 3, 12),     # more planes than workgroups
])
def test_clean_planes_matches_oracle(gpu, oracle, dt, n, ny, nx, per_psf, iters):
    from astroviper_amd.deconvolvers import hogbom as H
    n_psf = (n + per_psf - 1) // per_psf
    dirty, psf = _planes(n, ny, nx, n_psf, dt, n + ny + nx)
    r = torch.from_numpy(dirty.copy()).to(gpu)
    m = torch.zeros_like(r)
    # planes stop at different iterations
    thres = 2.2 if n == 300 else 0.0
    its = H.clean_planes_device(r, torch.from_numpy(psf).to(gpu), m, per_psf, iters, 0.3, thres)
    for p in range(0, n, 1 if n < 50 else 37):
        ref = oracle.hogbom_clean(dirty[p], psf[p // per_psf], max_iter=iters, gain=0.3,
                                  threshold=thres)
        assert its[p] == ref["iterations_performed"]
        np.testing.assert_array_equal(m[p].cpu().numpy(), ref["model_image"])
        np.testing.assert_array_equal(r[p].cpu().numpy(), ref["residual_image"])


@pytest.mark.parametrize("dt,n", [(np.float32, 2900), (np.float32, 4100), (np.float64, 2100)])
def test_clean_large_planes_match_oracle(gpu, oracle, dt, n):
    """Planes that need the most rows per lane, and one beyond the registers."""
    from astroviper_amd.deconvolvers import hogbom as H
    dirty, psf = _planes(1, n, n, 1, dt, n)
    r = torch.from_numpy(dirty.copy()).to(gpu)
    m = torch.zeros_like(r)
    its = H.clean_planes_device(r, torch.from_numpy(psf).to(gpu), m, 1, 6, 0.3, 0.0)
    ref = oracle.hogbom_clean(dirty[0], psf[0], max_iter=6, gain=0.3)
    assert its[0] == ref["iterations_performed"] == 6
    np.testing.assert_array_equal(m[0].cpu().numpy(), ref["model_image"])
    np.testing.assert_array_equal(r[0].cpu().numpy(), ref["residual_image"])


def test_clean_planes_refuses_mismatched_arrays(gpu):
    from astroviper_amd.deconvolvers import hogbom as H
    z = lambda *s: torch.zeros(s, device=gpu)  # noqa: E731
    with pytest.raises(ValueError):
        H.clean_planes_device(z(2, 8, 8), z(1, 8, 9), z(2, 8, 8), 2, 5)
    with pytest.raises(ValueError):
        H.clean_planes_device(z(4, 8, 8), z(1, 8, 8), z(4, 8, 8), 2, 5)
    assert H.clean_planes_device(z(0, 8, 8), z(1, 8, 8), z(0, 8, 8), 2, 5).size == 0
