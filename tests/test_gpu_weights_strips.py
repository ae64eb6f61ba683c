"""Imaging weights where a workgroup takes several strips of samples: the
channel changes inside a workgroup and inside a wavefront, the last block of
time steps is short and the last strip ragged; against the oracle."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

C = 299792458.0


# strips per workgroup: 1, 2 and 16 (one per 2048 strips of 256 samples, 16 at most)
@pytest.mark.parametrize("nt,nb,nchan", [(3, 1, 1), (5, 7, 3), (1501, 101, 7), (1500, 700, 8)])
def test_strips_match_oracle(gpu, oracle, nt, nb, nchan):
    from astroviper_amd.imaging_weighting.grid_imaging_weights import (degrid_imaging_weights,
                                                                       grid_imaging_weights)
    rng = np.random.default_rng(nt)
    n_uv = (90, 75)
    uvw = rng.uniform(-1500, 1500, size=(nt, nb, 3))
    uvw[1::2] = uvw[:-1:2]  # pairs of time steps share their pixels
    freq = np.linspace(1.0e9, 1.3e9, nchan)
    c = 0.5 * C / freq[-1] / 1300.0  # the longest fall off the grid
    w = rng.uniform(0.5, 1.5, size=(nt, nb, nchan, 1))
    w[rng.random(w.shape) < 0.1] = np.nan
    gp = {"image_size": n_uv, "cell_size": (-c, c)}
    g, s = np.zeros((nchan, 1) + n_uv), np.zeros((nchan, 1))
    grid_imaging_weights(g, s, uvw, w, freq, gp)
    gr, sr = np.zeros_like(g), np.zeros_like(s)
    oracle.grid_imaging_weights(gr, sr, uvw, w, freq, n_uv, (-c, c))
    # positive terms: the order of a sum of n changes it by n units at most
    np.testing.assert_allclose(s, sr, rtol=nt * nb * 2.0 ** -52)
    np.testing.assert_allclose(g, gr, rtol=nt * nb * 2.0 ** -52)
    bf = np.ones((2, nchan, 1))
    bf[0] = rng.uniform(0.5, 2.0, size=(nchan, 1))
    iw = degrid_imaging_weights(gr, uvw, w, bf, freq, gp)
    iwr = oracle.degrid_imaging_weights(gr, uvw, w, bf, freq, n_uv, (-c, c))
    # one product, sum and quotient per sample
    np.testing.assert_allclose(iw, iwr, rtol=4 * 2.0 ** -52)
