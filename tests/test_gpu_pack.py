"""The FP32 gridder over packed samples (one or two polarisations, 2^20 samples
or more, 16 x 16 tiles) against the FP64 oracle: flagged samples (with NaN and
infinite data), NaN and zero data and weights, no flags at all, either side of
2^20 samples, rows that carry their own channel and rows of two channels, and
samples that all reach four tiles, whose records leave no room to pack two
polarisations."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

C = 299792458.0
N_UV = (70, 96)


def data(n, n_pol, flags, rng):
    vis = (rng.normal(size=(n, n_pol)) + 1j * rng.normal(size=(n, n_pol))).astype(np.complex64)
    w = rng.uniform(0.5, 1.5, size=(n, n_pol)).astype(np.float32)
    flag = rng.random((n, n_pol)) < 0.3 if flags else np.zeros((n, n_pol), bool)
    vis[5:9, 0] = [np.nan, np.nan + 1j, 0, 1 + 1j * np.nan]
    w[9:12, -1] = [0.0, np.nan, 0.0]
    if flags:
        flag[20:24] = True
        vis[20:24, 0] = [np.nan, np.inf, 1, 1]
        w[23] = np.nan
    return vis, w, flag


def check(oracle, plan, vis, w, flag, flags, groups, uvw, freq, cell):
    """groups: per image channel (rows of vis / w / flag, rows of uvw)."""
    n, n_pol = vis.shape
    gref = np.zeros((len(groups), n_pol) + N_UV, complex)
    swref = np.zeros((len(groups), n_pol))
    for k, (m, rows) in enumerate(groups):
        wk = np.where(flag[m], 0.0, w[m].astype(np.float64))
        gk, sk = oracle.standard_grid(vis[m].astype(np.complex128).reshape(1, -1, 1, n_pol),
                                      uvw[rows].reshape(1, -1, 3), wk.reshape(1, -1, 1, n_pol),
                                      freq[k:k + 1], N_UV, cell, chan_mode="cube")
        gref[k], swref[k] = gk[0], sk[0]
    scale = np.max(np.abs(gref))
    assert scale > 0
    dev = plan.device
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    fl = to(flag.astype(np.uint8)) if flags else None
    g, sw = plan.grid(to(vis), to(w), fl)
    # FP32 sums of products of random signs: units in the last place of the
    # running sums, which wander to about the largest total
    assert np.max(np.abs(g.cpu().numpy() - gref)) < 1e-5 * scale
    np.testing.assert_allclose(sw.cpu().numpy(), swref, rtol=max(1e-12, n * 2.0 ** -53))
    # a second call adds the same again
    plan.grid(to(vis), to(w), fl, grid=g, sumwt=sw, accumulate=True)
    assert np.max(np.abs(g.cpu().numpy() - 2 * gref)) < 2e-5 * scale
    plan.close()


@pytest.mark.parametrize("flags", [True, False])
@pytest.mark.parametrize("n_pol", [1, 2])
@pytest.mark.parametrize("n", [257, (1 << 20) - 1, 1 << 20, (1 << 20) + 77])
def test_rows_with_their_own_channel(gpu, oracle, n, n_pol, flags):
    from astroviper_amd import device as D
    rng = np.random.default_rng(n)
    freq = np.array([1.0e9, 1.1e9, 1.3e9])
    chan = rng.integers(0, 3, size=n)
    uvw = rng.normal(scale=400.0, size=(n, 3))
    c = 0.3 * C / freq[-1] / 2000.0
    vis, w, flag = data(n, n_pol, flags, rng)
    dev = D.require_gpu()
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    plan = D.GridPlan(n, 3, 3, N_UV, (-c, c), tile=(16, 16), row_channels=True)
    plan.set_uvw(to(uvw), to(freq), row_chan=to(chan.astype(np.int32)))
    groups = [(chan == k, chan == k) for k in range(3)]
    check(oracle, plan, vis, w, flag, flags, groups, uvw, freq, (-c, c))


@pytest.mark.parametrize("n_pol", [1, 2])
@pytest.mark.parametrize("corners", [False, True])
def test_rows_of_channels(gpu, oracle, n_pol, corners):
    from astroviper_amd import device as D
    rng = np.random.default_rng(n_pol)
    rows, freq = (1 << 19) + 13, np.array([1.0e9, 1.0e9 + 1.0])
    c = 1e-4
    # positions in pixels; at the corners of tiles a footprint reaches four
    pos = (16.0 * rng.integers(1, 4, size=(rows, 2)) + rng.uniform(-0.5, 0.5, size=(rows, 2))
           if corners else rng.uniform(-2.0, 1.0, size=(rows, 2)) + rng.uniform(
               0, 1, size=(rows, 2)) * np.array(N_UV))
    uvw = np.zeros((rows, 3))
    for k, s in enumerate((-c, c)):
        uvw[:, k] = (pos[:, k] - N_UV[k] / 2) / (-s * N_UV[k]) * C / freq[0]
    vis, w, flag = data(2 * rows, n_pol, True, rng)
    dev = D.require_gpu()
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    plan = D.GridPlan(rows, 2, 2, N_UV, (-c, c), tile=(16, 16))
    plan.set_uvw(to(uvw), to(freq))
    if corners:
        assert plan.stats()["records"] > 3.9 * plan.stats()["grid_valid"] > 7.0 * rows
    groups = [(np.arange(2 * rows) % 2 == k, slice(None)) for k in range(2)]
    check(oracle, plan, vis, w, flag, True, groups, uvw, freq, (-c, c))
