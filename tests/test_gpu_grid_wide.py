"""The FP64 matrix-core gridder with workgroups of four wavefronts (few units)
and of eight (4096 or more): records in numbers that leave the last step, the
last four steps and the last wavefronts part empty, against the oracle."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

C = 299792458.0


@pytest.mark.parametrize("n_pol", [1, 2, 4])
@pytest.mark.parametrize("n_uv", [(96, 110), (1040, 1071)])
@pytest.mark.parametrize("n_time", [1, 13])
def test_fp64_gridder_matches_oracle(gpu, oracle, n_uv, n_pol, n_time):
    from astroviper_amd import device as D
    rng = np.random.default_rng(n_time)
    nb, nchan = 211, 3
    freq = np.linspace(1.0e9, 1.1e9, nchan)
    uvw = rng.normal(scale=300.0, size=(n_time, nb, 3))
    uvw[:, ::3] = uvw[:, :1] * 0.1  # a third of the samples crowd one bin
    c = 0.2 * C / freq[-1] / 1000.0 * np.array([-1.0, 1.0])
    shape = (n_time, nb, nchan, n_pol)
    vis = rng.normal(size=shape) + 1j * rng.normal(size=shape)
    w = rng.uniform(0.5, 1.5, size=shape)
    gref, swref = oracle.standard_grid(vis, uvw, w, freq, n_uv, tuple(c), chan_mode="cube")
    assert np.count_nonzero(gref) > 1000
    dev = D.require_gpu()
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    plan = D.GridPlan(n_time * nb, nchan, nchan, n_uv, tuple(c), n_baseline=nb)
    plan.set_uvw(to(uvw.reshape(-1, 3)), to(freq))
    g, sw = plan.grid(to(vis.reshape(-1, n_pol)), to(w.reshape(-1, n_pol)), None)
    # sums of at most a few hundred products in another order
    assert np.max(np.abs(g.cpu().numpy() - gref)) < 1e-12 * np.max(np.abs(gref))
    np.testing.assert_allclose(sw.cpu().numpy(), swref, rtol=1e-12)
    plan.close()
