"""How many segments the Mamba-1 scan cuts its rows into, read from the size of the scratch
that it asks for. The source of scratch refuses, so that nothing is launched; not run where
there is a GPU, on which a plan of whole rows (no scratch) would launch with the placeholder
pointers."""

import ctypes

import pytest

from armhackathon_amd import _ffi

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.skipif(torch.cuda.is_available(), reason="launches nothing: CPU only")


def _segments(batch, dim, length, state):
    lib = _ffi.load()
    asked = []

    def refuse(_, nbytes):
        asked.append(nbytes)
        return None

    alloc = _ffi.SCRATCH_ALLOC(refuse)
    at = ctypes.c_void_p(4096)  # an aligned address that nothing reads
    lib.arm_scan_thread_scratch(ctypes.cast(alloc, ctypes.c_void_p), None)
    try:
        rc = lib.arm_scan_selective_scan_f32(
            ctypes.byref(_ffi.ArmScanDims(batch, dim, length, state, 1)), at, at, at, at, at,
            None, None, None, 1, 0, 0, 0, at, None, None, None)
    finally:
        lib.arm_scan_thread_scratch(None, None)
    assert rc == 6 and len(asked) <= 1
    maps, rest = divmod(sum(asked), batch * dim * state * 2 * 4)
    assert rest == 0
    return maps + 1


@pytest.mark.parametrize("state,batch,dim,length,segments", [
    # the fastest of one to eight segments, or within 1% of it
    (16, 1, 1536, 2048, 8),
    (16, 2, 1536, 4096, 4),
    (16, 4, 1536, 2048, 1),
    (16, 3, 1536, 4096, 8),
    (64, 3, 1536, 8192, 8),
    # 256 row blocks of many states: eight segments in several rounds took 4 to 20% longer
    (64, 2, 2048, 4096, 3),
    (128, 2, 2048, 2048, 3),
    (128, 2, 2048, 4096, 3),
    # 224 blocks: eight took 6 to 19% longer
    (64, 1, 3584, 4096, 3),
    (128, 1, 3584, 2048, 3),
])
def test_segments_of_a_row(state, batch, dim, length, segments):
    assert _segments(batch, dim, length, state) == segments
