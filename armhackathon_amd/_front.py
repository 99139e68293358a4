"""Loads the native eager front-end (csrc/torch_front.cpp, built as _torch_front.so beside
libarm_scan_hip.so) and hands it the C ABI's functions.

`front()` is its module, for the public calls to try first: each of its functions serves
the plain eager call (float32 device tensors, no gradient, no transform or mode in
between) and returns None for any other, which then takes the custom op. It is None while
torch.compile traces, whose graphs hold the custom ops, and before the GPU is in use.
"""

import ctypes
import importlib.util
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

_module = None


def _load():
    global _module
    path = Path(__file__).resolve().parent / "_torch_front.so"
    if not path.is_file():
        raise OSError(f"{path} not found; build it with `make -C armhackathon_amd/csrc`")
    lib = _ffi.load()
    spec = importlib.util.spec_from_file_location(f"{__package__}._torch_front", path)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    module.bind({n: ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in _FUNCTIONS})
    _module = module
    return module


def front():
    if torch.compiler.is_compiling():
        return None
    if _module is not None:
        return _module
    return _load() if torch.cuda.is_initialized() else None
