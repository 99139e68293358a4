"""Where the native eager front-end cannot be had, the public calls take the custom ops, as
they did before it existed: no error of the loader's reaches the caller."""

import warnings

import pytest

from armhackathon_amd import _ffi, _front

torch = pytest.importorskip("torch")


class Without:
    """The library without some of its functions, as one of the same ABI version built
    before they were added."""

    ADDED = ("arm_scan_selective_scan_views_f32", "arm_scan_thread_scratch",
             "arm_scan_mamba3_grid_f32")

    def __init__(self, lib):
        self._lib = lib

    def __getattr__(self, name):
        if name in self.ADDED:
            raise AttributeError(name)
        return getattr(self._lib, name)


def test_older_library_is_declared():
    _ffi._declare(Without(_ffi.load()))


@pytest.mark.parametrize("why", ["missing", "not loadable", "older library", "other torch"])
def test_absent_front_end_leaves_the_custom_op(why, tmp_path, monkeypatch):
    import armhackathon_amd as arm_scan

    _ffi.load()
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: True)
    monkeypatch.setattr(_front, "_module", None)
    monkeypatch.setattr(_front, "_absent", False, raising=False)
    if why == "missing":
        monkeypatch.setattr(_front, "_PATH", tmp_path / "none.so")
    elif why == "not loadable":
        bad = tmp_path / "_torch_front.so"
        bad.write_bytes(b"not a library")
        monkeypatch.setattr(_front, "_PATH", bad)
    elif why == "older library":
        monkeypatch.setattr(_ffi, "_lib", Without(_ffi.load()))
    else:
        monkeypatch.setattr(torch, "__version__", "1.0.0+other")
    u = torch.zeros(1, 2, 8)
    bc = torch.zeros(1, 4, 8)
    with pytest.warns(RuntimeWarning, match="front-end is not in use"):
        with pytest.raises(ValueError, match="device tensors"):  # the custom op's refusal
            arm_scan.selective_scan(u, u, torch.zeros(2, 4), bc, bc)
    with warnings.catch_warnings():
        warnings.simplefilter("error")  # told once
        assert _front.front() is None


def test_missing_library_leaves_the_device(monkeypatch):
    """The loader's error comes before the call's device is made current."""
    from armhackathon_amd import op

    entered = []
    monkeypatch.setattr(torch.cuda.device, "__enter__", lambda self: entered.append(self))

    def missing():
        raise OSError("no library")

    monkeypatch.setattr(_ffi, "load", missing)
    with pytest.raises(OSError, match="no library"):
        with op._CaptureAware(torch.device("cuda", 0)):
            pass
    assert not entered
