"""Loads the native eager front-end (csrc/torch_front.cpp, built as _torch_front.so beside
this file) and hands it the C ABI's functions.

`front()` is its module, for the public calls to try first: each of its functions serves
the plain eager call (float32 device tensors, no gradient, no transform or mode in
between) and returns None for any other, which then takes the custom op. It is None while
torch.compile traces, whose graphs hold the custom ops, and before the GPU is in use.

The front-end is not needed: the custom ops run the same kernels. Where it is not there,
was built for another torch, or the library has not all the functions it calls, `front()`
is None for good, and one warning says why.
"""

import ctypes
import importlib.util
import warnings
from pathlib import Path

import torch

from . import _ffi

_FUNCTIONS = ("arm_scan_selective_scan_f32", "arm_scan_selective_scan_views_f32",
              "arm_scan_selective_state_update_f32",
              "arm_scan_selective_scan_bidirectional_f32",
              "arm_scan_mamba3_scan_time_major_f32", "arm_scan_mamba3_scan_angles_f32",
              "arm_scan_mamba3_scan_strided_f32", "arm_scan_mamba3_noncausal_f32",
              "arm_scan_mamba3_angles_f32", "arm_scan_mamba3_block_frontend_f32",
              "arm_scan_causal_conv1d_f32", "arm_scan_causal_conv1d_update_f32",
              "arm_scan_ss2d_f32", "arm_scan_mamba3_grid_f32", "arm_scan_thread_scratch")

_PATH = Path(__file__).resolve().parent / "_torch_front.so"
_module = None
_absent = False  # tried, and not to be had


def _load():
    """The front-end's module, bound to the library; raises where it cannot be had."""
    global _module
    if not _PATH.is_file():
        raise OSError(f"{_PATH} not found")
    lib = _ffi.load()
    missing = [n for n in _FUNCTIONS if not hasattr(lib, n)]
    if missing:
        raise OSError(f"{_ffi.lib_path()} does not export {', '.join(missing)}")
    spec = importlib.util.spec_from_file_location(f"{__package__}._torch_front", _PATH)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    built_for = getattr(module, "torch_version", None)
    if built_for != torch.__version__.split("+")[0]:
        raise ImportError(f"{_PATH} was built for torch {built_for}, this is "
                          f"{torch.__version__}")
    module.bind({n: ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in _FUNCTIONS})
    _module = module
    return module


def front():
    global _absent
    if torch.compiler.is_compiling():
        return None
    if _module is not None:
        return _module
    if _absent or not torch.cuda.is_initialized():
        return None
    _ffi.load()  # without the library nothing runs: its error is raised
    try:
        return _load()
    except (OSError, ImportError) as e:
        _absent = True
        warnings.warn(f"the native eager front-end is not in use ({e}); calls take the custom "
                      "ops, the same kernels at three times the host time. Rebuild with "
                      "`make -C armhackathon_amd/csrc`", RuntimeWarning, stacklevel=4)
        return None
