"""GPU binning where its passes change: one workgroup or several for the bin
offsets, chunks of one channel or of all, one or many chunks and segments,
and units shorter than a dense tile's records.

A misplaced, lost or doubled record is an O(1) error of the grid or the
model, so the FP64 bars of the parity tests (1e-12) apply."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

C = 299792458.0


def _rel(a, b):
    return float(np.max(np.abs(a - b)) / np.max(np.abs(b)))


def _samples(nt, nb, nchan, npol, n_uv, seed, spread=0.45):
    """Random uvw within `spread` of the grid's half width (some beyond it)."""
    rng = np.random.default_rng(seed)
    freq = np.linspace(1.0e9, 1.3e9, nchan)
    cell = 1e-4
    reach = spread * 2.2 * C / (2 * freq[-1] * cell)
    uvw = rng.uniform(-reach, reach, size=(nt, nb, 3))
    shape = (nt, nb, nchan, npol)
    vis = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    w = rng.uniform(0.5, 1.5, size=shape)
    flag = rng.random(shape) < 0.1
    return uvw, freq, vis, w, flag, (-cell, cell)


def _run(gpu, uvw, freq, vis, w, flag, n_uv, cell, cube, n_baseline, **plan_args):
    from astroviper_amd.device import GridPlan
    nt, nb, nchan, npol = w.shape
    rows = nt * nb
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)  # noqa: E731
    plan = GridPlan(rows, nchan, nchan if cube else 1, n_uv, cell, device=gpu,
                    n_baseline=n_baseline, **plan_args)
    plan.set_uvw(dev(uvw.reshape(rows, 3)), dev(freq))
    flat = (rows * nchan, npol)
    fl = dev(flag.reshape(flat).astype(np.uint8))
    g, sw = plan.grid(dev(vis.reshape(flat)), dev(w.reshape(flat)), fl)
    m = plan.degrid(g, fl)
    st = plan.stats()
    out = (g.cpu().numpy(), sw.cpu().numpy(), m.cpu().numpy(), st)
    plan.close()
    return out


# (times, baselines, channels, n_u, n_v, cube): bins = tiles x image channels
@pytest.mark.parametrize("nt,nb,nchan,n_u,n_v,cube", [
    (1, 1, 1, 16, 16, True),          # one bin, one sample
    (3, 21, 1, 64, 48, False),        # 63 rows: one partial mask word
    (4, 16, 4, 512, 512, True),       # 4096 bins: the last single-workgroup plan
    (4, 16, 4, 512, 528, True),       # 4224 bins: the general passes
    (40, 351, 4, 96, 112, False),     # chunks of all channels, rows in order
    (40, 351, 3, 96, 112, False),     # below the channels such chunks need
    (60, 45, 48, 160, 160, False),    # several chunks, runs of 48 channels
    (33, 67, 5, 1040, 1040, False),   # 4225 tiles: general passes, all channels
    (33, 67, 9, 1040, 1024, True),    # several blocks of bins per channel
])
def test_binning_paths_match_oracle(gpu, oracle, nt, nb, nchan, n_u, n_v, cube):
    n_uv = (n_u, n_v)
    uvw, freq, vis, w, flag, cell = _samples(nt, nb, nchan, 2, n_uv, nt * nb + nchan)
    w0 = np.where(flag, 0.0, w)
    gref, swref = oracle.standard_grid(vis, uvw, w0, freq, n_uv, cell,
                                       chan_mode="cube" if cube else "continuum")
    for n_baseline in (nb, 1):
        g, sw, m, st = _run(gpu, uvw, freq, vis, w, flag, n_uv, cell, cube, n_baseline)
        mref = oracle.degrid(uvw, flag, freq, gref, cell)
        if np.max(np.abs(gref)) > 0:
            assert _rel(g, gref) < 1e-12
            assert _rel(sw, swref) < 1e-12
            assert _rel(m.reshape(mref.shape), mref) < 1e-12
        assert st["grid_units"] >= st["bins"]


@pytest.mark.parametrize("cap", [64, 1024, 8192, 0])
@pytest.mark.parametrize("tile", [(16, 16), (32, 32), (24, 24)])
def test_compensated_sums_of_split_bins(gpu, oracle, cap, tile):
    """Compensated sums of bins of far more records than a unit holds (about
    20,000 per central tile) against the oracle.  Weights of one sign: a
    term's rounding (sample and table in FP32, one product each) stays below
    4 * 2^-24 of it, and 20,000 / 8192 groups add at most three roundings of
    the sum, so 8 * 2^-24 = 4.8e-7 of the largest cell bounds the error."""
    from astroviper_amd.device import GridPlan
    n_uv = (64, 64)
    nt, nb, nchan, npol = 120, 500, 2, 1
    uvw, freq, _, w, flag, cell = _samples(nt, nb, nchan, npol, n_uv, 5, spread=0.3)
    w = w.astype(np.float32)
    gref, swref = oracle.standard_grid(None, uvw, np.where(flag, 0, w).astype(float), freq, n_uv,
                                       cell, chan_mode="continuum", do_psf=True)
    rows = nt * nb
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)  # noqa: E731
    plan = GridPlan(rows, nchan, 1, n_uv, cell, tile=tile, unit_cap=cap, device=gpu)
    plan.set_uvw(dev(uvw.reshape(rows, 3)), dev(freq))
    g, sw = plan.grid(None, dev(w.reshape(-1, npol)),
                      dev(flag.reshape(-1, npol).astype(np.uint8)), psf=True, compensated=True)
    assert _rel(g.cpu().numpy(), gref) < 8 * 2.0 ** -24
    assert _rel(sw.cpu().numpy(), swref) < 1e-12
    # accumulating the same samples doubles the grid
    g2, sw2 = plan.grid(None, dev(w.reshape(-1, npol)),
                        dev(flag.reshape(-1, npol).astype(np.uint8)), grid=g, sumwt=sw, psf=True,
                        accumulate=True, compensated=True)
    assert _rel(g2.cpu().numpy(), 2 * gref) < 16 * 2.0 ** -24
    assert _rel(sw2.cpu().numpy(), 2 * swref) < 1e-12
    plan.close()


@pytest.mark.parametrize("chan_map,n_img", [
    ([2, 0, 1, 4, 3], 5),          # a permutation
    ([1, 1, 0, 0, 2, 1, 2], 3),    # channels averaged into three
    ([0, -1, 0, 5, 0], 1),         # some mapped outside the grid
    ([3, 0, 0, 6, 1, 2, 5, 4], 8),  # as many image channels, not one to one
])
@pytest.mark.parametrize("n_u", [96, 1040])
def test_channel_maps(gpu, oracle, chan_map, n_img, n_u):
    from astroviper_amd.device import GridPlan
    nt, nb, nchan, n_uv = 6, 67, len(chan_map), (n_u, n_u)
    uvw, freq, vis, w, flag, cell = _samples(nt, nb, nchan, 1, n_uv, 17)
    cube, sw = oracle.standard_grid(vis, uvw, np.where(flag, 0, w), freq, n_uv, cell,
                                    chan_mode="cube")
    gref = np.zeros((n_img,) + cube.shape[1:], dtype=complex)
    swref = np.zeros((n_img, 1))
    for c, ic in enumerate(chan_map):
        if 0 <= ic < n_img:
            gref[ic] += cube[c]
            swref[ic] += sw[c]
    rows = nt * nb
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)  # noqa: E731
    plan = GridPlan(rows, nchan, n_img, n_uv, cell, device=gpu, n_baseline=nb)
    plan.set_uvw(dev(uvw.reshape(rows, 3)), dev(freq), dev(np.array(chan_map, dtype=np.int32)))
    g, s = plan.grid(dev(vis.reshape(-1, 1)), dev(w.reshape(-1, 1)),
                     dev(flag.reshape(-1, 1).astype(np.uint8)))
    assert _rel(g.cpu().numpy(), gref) < 1e-12
    assert _rel(s.cpu().numpy(), swref) < 1e-12
    plan.close()


@pytest.mark.parametrize("n_rows,order", [(1, "sorted"), (63, "mixed"), (5000, "sorted"),
                                          (5000, "mixed"), (1 << 21, "sorted")])
def test_rows_with_their_own_channel(gpu, oracle, n_rows, order):
    """Blocks of rows of one channel, of several, and of out-of-range ones."""
    from astroviper_amd.device import GridPlan
    rng = np.random.default_rng(n_rows)
    n_uv, nchan, cell = (96, 112), 5, (-1e-4, 1e-4)
    freq = np.linspace(1.0e9, 1.3e9, nchan)
    uvw = rng.uniform(-1100.0, 1100.0, size=(n_rows, 3))
    chan = rng.integers(-1, nchan + 1, size=n_rows)
    if order == "sorted":
        chan = np.sort(chan)
    vis = rng.standard_normal(n_rows) + 1j * rng.standard_normal(n_rows)
    w = rng.uniform(0.5, 1.5, size=n_rows)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)  # noqa: E731
    plan = GridPlan(n_rows, nchan, nchan, n_uv, cell, device=gpu, row_channels=True)
    plan.set_uvw(dev(uvw), dev(freq), None, dev(chan.astype(np.int32)))
    g, s = plan.grid(dev(vis.reshape(-1, 1)), dev(w.reshape(-1, 1)))
    m = plan.degrid(g).cpu().numpy()[:, 0]
    g, s = g.cpu().numpy(), s.cpu().numpy()
    plan.close()
    for c in range(nchan):
        r = chan == c
        if not r.any():
            assert not g[c].any()
            continue
        shape = (1, int(r.sum()), 1, 1)
        gref, sref = oracle.standard_grid(vis[r].reshape(shape), uvw[r].reshape(1, -1, 3),
                                          w[r].reshape(shape), freq[c:c + 1], n_uv, cell,
                                          chan_mode="cube")
        if np.abs(gref).max() > 0:
            assert _rel(g[c], gref[0]) < 1e-12 and _rel(s[c], sref[0]) < 1e-12
            mref = oracle.degrid(uvw[r].reshape(1, -1, 3), np.zeros(shape, bool), freq[c:c + 1],
                                 gref, cell)
            assert _rel(m[r], mref.ravel()) < 1e-12
    assert not m[(chan < 0) | (chan >= nchan)].any()


@pytest.mark.parametrize("cap,per_tile,npol", [
    (3000, 6500, 1), (3000, 6500, 2), (5000, 6500, 1), (6000, 6500, 4), (100, 8150, 1),
    (8191, 8192, 1), (4096, 8193, 1),
])
def test_compensated_sums_of_neighbouring_split_bins(gpu, oracle, cap, per_tile, npol):
    """Unit caps that do not divide the records of a compensated group, on
    neighbouring tiles of equally many records, each in one tile only: a tile
    that took another's sums would be off by its own size.  The sums are of
    terms of one sign, in two groups at most: the bound of the test above."""
    from astroviper_amd.device import GridPlan
    n, tiles = 64, 16
    rng = np.random.default_rng(cap + npol)
    # 4 pixels about every tile's centre: footprints of 7 stay inside
    at = np.repeat(np.arange(tiles), per_tile)
    px = np.stack([16 * (at // 4), 16 * (at % 4)], 1) + 8 + rng.uniform(-4, 4, (at.size, 2))
    px = px[rng.permutation(at.size)]
    freq, cell = np.array([1.2e9]), 1e-4
    scale = -(freq[0] * np.array([-cell, cell]) * n) / C
    uvw = np.concatenate([(px - n // 2) / scale, np.zeros((at.size, 1))], 1)
    w = rng.uniform(0.5, 1.5, (at.size, npol)).astype(np.float32)
    gref, swref = oracle.standard_grid(None, uvw[:, None], w[:, None, None].astype(float), freq,
                                       (n, n), (-cell, cell), chan_mode="cube", do_psf=True)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)  # noqa: E731
    plan = GridPlan(at.size, 1, 1, (n, n), (-cell, cell), unit_cap=cap, device=gpu)
    plan.set_uvw(dev(uvw), dev(freq))
    st = plan.stats()
    assert st["records"] == tiles * per_tile and st["bins"] == tiles
    g, sw = plan.grid(None, dev(w), psf=True, compensated=True)
    assert _rel(g.cpu().numpy(), gref) < 8 * 2.0 ** -24
    assert _rel(sw.cpu().numpy(), swref) < 1e-12
    g, sw = plan.grid(None, dev(w), grid=g, sumwt=sw, psf=True, accumulate=True, compensated=True)
    assert _rel(g.cpu().numpy(), 2 * gref) < 16 * 2.0 ** -24
    plan.close()


@pytest.mark.parametrize("nt,nb,nchan,n,cube", [
    (5, 512, 3, 80, True),      # chunks of 1024 rows: rows in order
    (5, 1536, 2, 1040, True),   # chunks of 3072 rows: two time steps, then a part
    (5, 1537, 2, 1040, True),   # one row fewer than two
    (9, 33, 31, 80, False),     # all channels of 66 rows and more, 31 and 32
    (9, 33, 32, 80, False),
    (40, 32, 31, 528, False),
])
def test_binning_of_few_time_steps_a_chunk(gpu, oracle, nt, nb, nchan, n, cube):
    n_uv = (n + 16, n)
    uvw, freq, vis, w, flag, cell = _samples(nt, nb, nchan, 1, n_uv, nb + nchan)
    gref, swref = oracle.standard_grid(vis, uvw, np.where(flag, 0.0, w), freq, n_uv, cell,
                                       chan_mode="cube" if cube else "continuum")
    g, sw, m, st = _run(gpu, uvw, freq, vis, w, flag, n_uv, cell, cube, nb)
    mref = oracle.degrid(uvw, flag, freq, gref, cell)
    assert _rel(g, gref) < 1e-12 and _rel(sw, swref) < 1e-12
    assert _rel(m.reshape(mref.shape), mref) < 1e-12


@pytest.mark.parametrize("nchan", [1, 2, 4])
@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_degrid_units_longer_than_grid_units(gpu, nchan, prec):
    """Plans of samples enough for degrid caps of two and four grid caps: a
    sample's sum does not depend on its unit, so one cap for both gives the same
    bits, on bins of many units and of one."""
    from astroviper_amd.device import GridPlan
    cdt = torch.complex64 if prec == "fp32" else torch.complex128
    n, nb, nt = 112, 350, 1 + 1_300_000 // (350 * nchan)
    uvw, freq, _, _, _, cell = _samples(nt, nb, nchan, 1, (n, n), nchan, spread=0.3)
    gen = torch.Generator(device=gpu).manual_seed(nchan)
    grid = torch.randn((nchan, 2, n, n), generator=gen, device=gpu, dtype=cdt)
    out, units = [], []
    for cap in (0, 8192, 64):
        plan = GridPlan(nt * nb, nchan, nchan, (n, n), cell, unit_cap=cap, device=gpu,
                        n_baseline=nb)
        plan.set_uvw(torch.from_numpy(uvw.reshape(-1, 3)).to(gpu), torch.from_numpy(freq).to(gpu))
        out.append(plan.degrid(grid))
        units.append((plan.stats()["grid_units"], plan.stats()["degrid_units"]))
        plan.close()
    assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])
    assert float(out[0].abs().max()) > 0
    # 256 records a grid unit; as many, two and four times as many a degrid unit
    ratio = units[0][0] / units[0][1]
    assert ratio > {1: 1.0, 2: 1.8, 4: 3.0}[nchan]


@pytest.mark.parametrize("npol", [1, 2, 4])
@pytest.mark.parametrize("cap", [0, 64, 100, 4096, 8192])
@pytest.mark.parametrize("n", [80, 1040])
def test_compensated_sums_of_few_and_many_split_bins(gpu, oracle, n, cap, npol):
    """Bins of one unit, of two, of several and of several groups, side by side
    on a plan where most bins are split (80^2: 25 tiles) and on one where few
    are (1040^2: 4225), the sums and their bounds as above."""
    from astroviper_amd.device import GridPlan
    tiles = (n // 16) ** 2
    counts = np.full(tiles, 3)
    counts[:8] = (13000, 9000, 5000, 700, 200, 150, 520, 64)
    counts[-2:] = (8300, 129)
    rng = np.random.default_rng(n + cap + npol)
    at = np.repeat(np.arange(tiles), counts)
    nt = n // 16
    px = np.stack([16 * (at // nt), 16 * (at % nt)], 1) + 8 + rng.uniform(-4, 4, (at.size, 2))
    px = px[rng.permutation(at.size)]
    freq, cell = np.array([1.2e9]), 1e-4
    scale = -(freq[0] * np.array([-cell, cell]) * n) / C
    uvw = np.concatenate([(px - n // 2) / scale, np.zeros((at.size, 1))], 1)
    w = rng.uniform(0.5, 1.5, (at.size, npol)).astype(np.float32)
    gref, swref = oracle.standard_grid(None, uvw[:, None], w[:, None, None].astype(float), freq,
                                       (n, n), (-cell, cell), chan_mode="cube", do_psf=True)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)  # noqa: E731
    plan = GridPlan(at.size, 1, 1, (n, n), (-cell, cell), unit_cap=cap, device=gpu)
    plan.set_uvw(dev(uvw), dev(freq))
    assert plan.stats()["records"] == at.size
    g, sw = plan.grid(None, dev(w), psf=True, compensated=True)
    assert _rel(g.cpu().numpy(), gref) < 8 * 2.0 ** -24
    assert _rel(sw.cpu().numpy(), swref) < 1e-12
    # small bins by themselves: beside the largest cell their errors would not show
    tail = np.s_[..., -32:-16, :]
    assert _rel(g.cpu().numpy()[tail], gref[tail]) < 8 * 2.0 ** -24
    g, sw = plan.grid(None, dev(w), grid=g, sumwt=sw, psf=True, accumulate=True, compensated=True)
    assert _rel(g.cpu().numpy(), 2 * gref) < 16 * 2.0 ** -24
    plan.close()
