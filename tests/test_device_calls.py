"""How the Python layer makes its device calls, without a GPU: the library's
entry points are replaced, so tensors stay on the CPU."""
import weakref

import numpy as np
import pytest

torch = pytest.importorskip("torch")

AX = (-2, -1)


def test_copies_for_a_call_live_until_it_is_made(monkeypatch):
    """An operand copied for its alignment or layout is still held when the
    library is called: freed before, another thread's tensor could take its
    memory on the same stream."""
    from astroviper_amd import device as D
    passed, alive = [], []
    monkeypatch.setattr(D, "_aligned", lambda t, n: None if t is None else t.clone())
    monkeypatch.setattr(D, "_ptr", lambda t: None if t is None else passed.append(weakref.ref(t)))
    monkeypatch.setattr(D, "_stream", lambda: None)
    monkeypatch.setattr(D, "call", lambda *a: alive.append(all(t() is not None for t in passed)))
    g = torch.zeros((1, 1, 8, 8), dtype=torch.complex64)
    x = torch.zeros((1, 1, 8, 8))
    work = torch.zeros(1, dtype=torch.uint8)
    D.uv_to_image(g, None, x.clone(), work)
    passed.clear()
    D.image_to_uv(x, g.clone(), work)
    passed.clear()
    plan = object.__new__(D.GridPlan)
    plan.n_rows, plan.n_chan, plan.row_chan, plan._h = 4, 1, None, None
    plan.device, plan.cgk = torch.device("cpu"), torch.zeros(3)
    plan.degrid(g.transpose(-1, -2), torch.zeros((4, 1), dtype=torch.bool))
    passed.clear()
    plan.n_img_chan, plan.n_u, plan.n_v = 1, 8, 8
    plan.grid(torch.zeros((4, 1), dtype=torch.complex64), torch.ones((4, 1)))
    assert alive == [True] * 4


@pytest.mark.parametrize("shape", [(2, 18, 30), (3, 2, 50, 36), (1, 6, 10)])
def test_model_to_uv_on_the_host(shape):
    """Even axes that are no multiples of 4 are transformed by torch wherever
    the model lies, with its gradient, as any tensor function."""
    from astroviper_amd.major_cycle import model_to_uv
    rng = np.random.default_rng(sum(shape))
    x = rng.standard_normal(shape)
    ref = np.fft.fftshift(np.fft.fft2(np.fft.ifftshift(x, axes=AX), axes=AX), axes=AX)
    t = torch.from_numpy(x).requires_grad_(True)
    uv = model_to_uv(t, torch.complex128)
    # two FP64 transforms of a few hundred points: a few roundings of the largest
    np.testing.assert_allclose(uv.detach().numpy(), ref, rtol=0, atol=1e-13 * np.abs(ref).max())
    torch.view_as_real(uv).square().sum().backward()
    grad = 2 * shape[-2] * shape[-1] * x
    np.testing.assert_allclose(t.grad.numpy(), grad, rtol=0, atol=1e-13 * np.abs(grad).max())


def _fake_clean(monkeypatch, H, planes):
    """clean_planes_device with a library call that fills its arguments by
    `planes(result, work)`; the real one's records and header."""
    def call(name, *args):
        assert name == "av_hogbom_clean_planes"
        planes(args[11].view(torch.int32).reshape(-1, 6), args[12].view(torch.int32))

    monkeypatch.setattr(H._lib, "call", call)
    monkeypatch.setattr(H._dev, "_ptr", lambda t: t)
    monkeypatch.setattr(H._dev, "_stream", lambda: None)
    r = torch.zeros((3, 8, 8))
    # a buffer of another call before
    work = torch.full((4096,), 7, dtype=torch.uint8)
    return H.clean_planes_device(r, torch.ones((3, 8, 8)), torch.zeros_like(r), 1, 5, work=work)


def test_a_missed_exchange_is_reported(monkeypatch):
    """A workgroup that gives up leaves its mark in the work's header even
    where every plane's record was written by one that did not."""
    from astroviper_amd import _lib
    from astroviper_amd.deconvolvers import hogbom as H

    def done(result, work):
        work[:16] = 0
        result[:] = 0
        result[:, 0] = 5

    assert _fake_clean(monkeypatch, H, done).tolist() == [5, 5, 5]

    def late(result, work):
        done(result, work)
        work[1] = 1

    with pytest.raises(_lib.AvgridError):
        _fake_clean(monkeypatch, H, late)

    def one_plane(result, work):
        done(result, work)
        result[2, 3] = -1

    with pytest.raises(_lib.AvgridError):
        _fake_clean(monkeypatch, H, one_plane)
