"""Host arrays to the device and back through page-locked chunks (below the
size copied straight, at one, two and more chunks, with a ragged last one),
arrays a chunked copy does not take, and the stager's buffers when a longer
partition follows a short one."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbytes", [0, 40, (1 << 20) - 8, 1 << 20, (8 << 20) - 8, 8 << 20,
                                    (8 << 20) + 8, 16 << 20, (24 << 20) + 16, (32 << 20) + 8])
def test_upload_download(gpu, nbytes):
    from astroviper_amd import device as D
    a = np.random.default_rng(nbytes).standard_normal(nbytes // 8)
    t = D.upload(a, D.require_gpu())
    a_then, a[:] = a.copy(), np.nan  # the source is free once upload returns
    np.testing.assert_array_equal(t.cpu().numpy(), a_then)
    out = np.empty_like(a)
    D.download(t * 2, out)
    np.testing.assert_array_equal(out, 2 * a_then)


def test_download_forms(gpu):
    from astroviper_amd import device as D
    rng = np.random.default_rng(0)
    a = (rng.standard_normal((3, 700, 901)) + 1j * rng.standard_normal((3, 700, 901)))
    t = D.upload(a, D.require_gpu())
    for out in (np.empty(a.shape, np.complex128), np.empty(a.shape, np.complex64),
                np.empty(a.shape[::-1], np.complex128).T, np.empty((2,) + a.shape, a.dtype)[1]):
        D.download(t, out)
        np.testing.assert_array_equal(out, a.astype(out.dtype))
    out = np.empty(a.shape[::-1], a.dtype)
    D.download(t.conj().permute(2, 1, 0), out)  # lazily conjugated, not contiguous
    np.testing.assert_array_equal(out, a.conj().T)
    out = np.empty(a.shape)
    D.download(t.real, out)
    np.testing.assert_array_equal(out, a.real)


@pytest.mark.parametrize("n_time,block", [((3, 9, 2), 4), ((2, 3), 100), ((5, 2, 6), 5)])
def test_stager_grows(gpu, oracle, n_time, block):
    from test_gpu_staging import oracle_grid, partitions, rel
    from astroviper_amd import staging as S
    parts, n_uv, cell = partitions(n_time)
    gref, swref = oracle_grid(oracle, parts, n_uv, cell, "cube")
    ps = [S.array_partition(p["vis"], p["uvw"], p["w"], p["flag"], p["freq"]) for p in parts]
    g, sw = S.grid_processing_set(ps, n_uv, cell, chan_mode="cube", fp32=False,
                                  block_rows=block * parts[0]["w"].shape[1])
    assert rel(g.cpu().numpy(), gref) < 1e-12
    np.testing.assert_allclose(sw.cpu().numpy(), swref, rtol=1e-12)
