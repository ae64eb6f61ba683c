"""The FP64 degridder with two polarisations, whose records are split by v
where both halves' windows hold every footprint (supports up to 7 in tiles 16
wide) and not beyond, against the oracle: samples crowded into one half of a
tile, on the columns either side of the split, and at the grid's edges."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

C = 299792458.0


@pytest.mark.parametrize("support", [2, 3, 6, 7, 8])
@pytest.mark.parametrize("tile,n_uv", [((16, 16), (75, 90)), ((48, 16), (130, 64)),
                                       ((16, 8), (64, 50))])
def test_fp64_two_polarisations_match_oracle(gpu, oracle, support, tile, n_uv):
    from astroviper_amd import device as D
    rng = np.random.default_rng(support)
    nt, nb, ov = 3, 300, 20
    freq = np.array([1.0e9, 1.2e9])
    cell = (-1e-4, 1.3e-4)
    # positions in pixels of the first channel, from edge to edge
    pos = rng.uniform(0, 1, size=(nt, nb, 2)) * np.array(n_uv)
    pos[0, :100, 1] = 16 + rng.uniform(6.0, 9.0, size=100)   # about the split of one tile
    pos[1, :40] = 20 + rng.uniform(0.0, 1.0, size=(40, 2))   # one half only
    uvw = np.zeros((nt, nb, 3))
    for k in range(2):
        uvw[..., k] = (n_uv[k] / 2 - pos[..., k]) / (cell[k] * n_uv[k]) * C / freq[0]
    flag = rng.random((nt, nb, 2, 2)) < 0.1
    grid = rng.normal(size=(2, 2) + n_uv) + 1j * rng.normal(size=(2, 2) + n_uv)
    mref = oracle.degrid(uvw, flag, freq, grid, cell, support=support, sampling=ov)
    assert np.count_nonzero(mref) > 1000
    dev = D.require_gpu()
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    plan = D.GridPlan(nt * nb, 2, 2, n_uv, cell, support, ov, tile=tile)
    plan.set_uvw(to(uvw.reshape(-1, 3)), to(freq))
    m = plan.degrid(to(grid), to(flag.reshape(-1, 2).astype(np.uint8))).cpu().numpy()
    # a sum of support^2 terms over the sum of their weights
    assert np.max(np.abs(m.reshape(mref.shape) - mref)) < 1e-12 * np.max(np.abs(mref))
    plan.close()
