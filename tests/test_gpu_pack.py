"""Gridding a plan whose rows carry their own channel, with one polarisation
in FP32 16 x 16 tiles (their samples packed side by side first), against the
FP64 oracle: flagged samples (with NaN and infinite data), NaN and zero data and
weights, no flags at all, either side of the 2^20 rows from which they are."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

C = 299792458.0


@pytest.mark.parametrize("flags", [True, False])
@pytest.mark.parametrize("n", [257, (1 << 20) - 1, 1 << 20, (1 << 20) + 77])
def test_packed_rows_match_oracle(gpu, oracle, n, flags):
    from astroviper_amd import device as D
    rng = np.random.default_rng(n)
    n_uv, nchan = (70, 96), 3
    freq = np.array([1.0e9, 1.1e9, 1.3e9])
    chan = rng.integers(0, nchan, size=n)
    uvw = rng.normal(scale=400.0, size=(n, 3))
    c = 0.3 * C / freq[-1] / 2000.0
    vis = (rng.normal(size=n) + 1j * rng.normal(size=n)).astype(np.complex64)
    w = rng.uniform(0.5, 1.5, size=n).astype(np.float32)
    flag = rng.random(n) < 0.3 if flags else np.zeros(n, bool)
    vis[5:9] = [np.nan, np.nan + 1j, 0, 1 + 1j * np.nan]
    w[9:12] = [0.0, np.nan, 0.0]
    if flags:
        flag[20:24] = True
        vis[20:24] = [np.nan, np.inf, 1, 1]
        w[23] = np.nan
    gref = np.zeros((nchan, 1) + n_uv, complex)
    swref = np.zeros((nchan, 1))
    for k in range(nchan):  # the oracle takes whole channels: a row's own only
        m = chan == k
        if not m.any():
            continue
        wk = np.where(flag[m], 0.0, w[m].astype(np.float64))
        vk = vis[m].astype(np.complex128)
        gk, sk = oracle.standard_grid(vk.reshape(1, -1, 1, 1), uvw[m].reshape(1, -1, 3),
                                      wk.reshape(1, -1, 1, 1), freq[k:k + 1], n_uv, (-c, c),
                                      chan_mode="cube")
        gref[k], swref[k] = gk[0], sk[0]
    dev = D.require_gpu()
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    plan = D.GridPlan(n, nchan, nchan, n_uv, (-c, c), tile=(16, 16), row_channels=True)
    plan.set_uvw(to(uvw), to(freq), row_chan=to(chan.astype(np.int32)))
    fl = to(flag.astype(np.uint8)[:, None]) if flags else None
    g, sw = plan.grid(to(vis[:, None]), to(w[:, None]), fl)
    # FP32 sums of products of random signs: units in the last place of the
    # running sums, which wander to about the largest total
    scale = max(np.max(np.abs(gref)), 1e-30)
    assert np.max(np.abs(g.cpu().numpy() - gref)) < 1e-5 * scale
    np.testing.assert_allclose(sw.cpu().numpy(), swref, rtol=max(1e-12, n * 2.0 ** -53))
    # a second call adds the same again
    plan.grid(to(vis[:, None]), to(w[:, None]), fl, grid=g, sumwt=sw, accumulate=True)
    assert np.max(np.abs(g.cpu().numpy() - 2 * gref)) < 2e-5 * scale
    plan.close()
