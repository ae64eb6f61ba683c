"""The fused FFTs between uv grids and real images (av_uv_to_image,
av_image_to_uv) against NumPy's shifted FFTs in FP64, over axes of every radix
and mix of them, few and many rows and columns of a workgroup, planes of
several groups, and the sizes torch.fft keeps.

An FFT's relative error (2-norm) grows as a small multiple of 2^-53 log2(n);
1e-14 bounds it with a wide margin, 4 * 2^-24 where a type in memory is FP32."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

AX = (-2, -1)
# every radix first and last, one pass more or less, one workgroup or many
SIZES = [(16, 32), (10, 20), (12, 18), (18, 12), (30, 50), (64, 48), (96, 250), (486, 54),
         (240, 1024), (1024, 240), (1500, 100), (2048, 64), (2050 - 2, 36), (4096, 32), (20, 4000),
         (24, 16384), (54, 5000)]


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def _taper(oracle, n, m):
    return oracle.create_prolate_spheroidal_kernel(100, 7, np.array([n, m]))[1]


@pytest.mark.parametrize("n,m", SIZES)
def test_uv_to_image_matches_shifted_ifft(gpu, oracle, n, m):
    from astroviper_amd import device as D
    rng = np.random.default_rng(n * 7 + m)
    planes = 3 if n * m < 1 << 18 else 2
    g = rng.standard_normal((planes, n, m)) + 1j * rng.standard_normal((planes, n, m))
    sw = rng.uniform(1, 9, size=planes)
    taper = _taper(oracle, n, m)
    for cdt, tol in ((np.complex128, 1e-14), (np.complex64, 1e-14)):
        gt = g.astype(cdt)
        ref = np.fft.fftshift(np.fft.ifft2(np.fft.ifftshift(gt.astype(complex), axes=AX),
                                           axes=AX), axes=AX).real * (n * m)
        t = torch.from_numpy(gt).to(gpu)
        work = D.fft_work(planes, n, m, gpu)
        assert work is not None
        for odt, otol in ((torch.float64, tol), (torch.float32, 4 * 2.0 ** -24)):
            out = torch.empty((planes, n, m), dtype=odt, device=gpu)
            D.uv_to_image(t, torch.from_numpy(sw).to(gpu), out, work)
            assert _rel(out.cpu().numpy() * taper * sw[:, None, None], ref) < otol
            D.uv_to_image(t, None, out, work, taper=False)
            assert _rel(out.cpu().numpy(), ref) < otol


@pytest.mark.parametrize("n,m", SIZES)
def test_image_to_uv_matches_shifted_fft(gpu, oracle, n, m):
    from astroviper_amd import device as D
    rng = np.random.default_rng(n * 5 + m)
    planes = 3 if n * m < 1 << 18 else 2
    x = rng.standard_normal((planes, n, m))
    taper = _taper(oracle, n, m)
    for xdt in (np.float64, np.float32):
        xt = x.astype(xdt)
        for cdt, tol in ((torch.complex128, 1e-14), (torch.complex64, 4 * 2.0 ** -24)):
            work = D.fft_work(planes, n, m, gpu)
            for tp in (False, True):
                xx = xt.astype(float) / (taper if tp else 1.0)
                ref = np.fft.fftshift(np.fft.fft2(np.fft.ifftshift(xx, axes=AX), axes=AX),
                                      axes=AX)
                out = torch.empty((planes, n, m), dtype=cdt, device=gpu)
                D.image_to_uv(torch.from_numpy(xt).to(gpu), out, work, taper=tp)
                assert _rel(out.cpu().numpy(), ref) < tol


def test_fft_groups_of_planes(gpu):
    """More planes than a group holds, against torch plane by plane."""
    from astroviper_amd import device as D
    n, planes = 1024, 270  # 8.4 MB of half spectrum a plane
    gen = torch.Generator(device=gpu).manual_seed(3)
    g = torch.randn((planes, n, n), generator=gen, device=gpu, dtype=torch.complex64)
    work = D.fft_work(planes, n, n, gpu)
    assert work.numel() < planes * n * (n // 2 + 1) * 16
    out = D.uv_to_image(g, None, torch.empty((planes, n, n), dtype=torch.float64, device=gpu), work,
                        taper=False)
    for p in (0, 1, 100, 253, 254, 255, 256, planes - 1):  # 255 planes are a group
        ref = torch.fft.fftshift(torch.fft.ifft2(torch.fft.ifftshift(g[p].to(torch.complex128)))
                                 ).real * (n * n)
        assert float((out[p] - ref).norm() / ref.norm()) < 1e-14
    back = D.image_to_uv(out, torch.empty((planes, n, n), dtype=torch.complex128, device=gpu),
                         work)
    for p in (0, planes - 1):
        ref = torch.fft.fftshift(torch.fft.fft2(torch.fft.ifftshift(out[p])))
        assert float((back[p] - ref).norm() / ref.norm()) < 1e-14


def test_fft_sizes_left_to_torch(gpu):
    from astroviper_amd import device as D
    for n, m in ((15, 16), (16, 15), (14, 16), (16, 28), (22, 22), (8192, 16), (2, 16), (16, 4)):
        assert D.fft_work(1, n, m, gpu) is None
    with pytest.raises(NotImplementedError):
        D.uv_to_image(torch.zeros((14, 16), dtype=torch.complex64, device=gpu), None,
                      torch.zeros((14, 16), device=gpu),
                      torch.zeros(1 << 16, dtype=torch.uint8, device=gpu))
    # a view off the alignment of the loads
    g = torch.randn(16 * 32 + 1, device=gpu, dtype=torch.complex64)[1:].reshape(16, 32)
    work = D.fft_work(1, 16, 32, gpu)
    a = D.uv_to_image(g, None, torch.empty((16, 32), device=gpu), work)
    b = D.uv_to_image(g.clone(), None, torch.empty((16, 32), device=gpu), work)
    assert torch.equal(a, b)


@pytest.mark.parametrize("odt,tol", [(torch.float64, 1e-14), (torch.float32, 4 * 2.0 ** -24)])
def test_sums_of_weights_without_taper(gpu, odt, tol):
    """1 / sumwt and the taper are independent of each other."""
    from astroviper_amd import device as D
    n, m, planes = 30, 48, 3
    rng = np.random.default_rng(4)
    g = rng.standard_normal((planes, n, m)) + 1j * rng.standard_normal((planes, n, m))
    sw = rng.uniform(2, 9, size=planes)
    ref = np.fft.fftshift(np.fft.ifft2(np.fft.ifftshift(g, axes=AX), axes=AX), axes=AX).real * n * m
    out = torch.empty((planes, n, m), dtype=odt, device=gpu)
    D.uv_to_image(torch.from_numpy(g).to(gpu), torch.from_numpy(sw).to(gpu), out,
                  D.fft_work(planes, n, m, gpu), taper=False)
    assert _rel(out.cpu().numpy(), ref / sw[:, None, None]) < tol
