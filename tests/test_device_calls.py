"""How the Python layer makes its device calls, without a GPU: the library's
entry points are replaced, so tensors stay on the CPU."""
import pytest

torch = pytest.importorskip("torch")


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
