"""A library of the same ABI version without the functions that only the native eager
front-end calls is declared and used, as it was before they were added."""

from armhackathon_amd import _ffi


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
