"""The width-4 time-major convolution (a thread's run of 4 or 16 steps of four channels)
against the tile kernel's contiguous output, which is checked against numpy in
test_m1_gpu.py: the same taps in the same order, so the same bits. Lengths around the
runs, small and large calls, and inputs whose pieces are not aligned."""

import pytest

from util import case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 4, 1), (2, 8, 3), (1, 36, 5), (3, 1536, 77),
                                   (1, 1536, 4097), (8, 1536, 1023)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("act", [None, "silu"])
def test_time_major_bits(shape, offset, act):
    import torch

    import armhackathon_amd as arm

    b, d, L = shape
    case(f"conv time-major {shape} offset {offset} {act}")
    gen = torch.Generator(device="cuda").manual_seed(L)
    wide = torch.randn(b * L * 2 * d + offset, device="cuda", generator=gen)[offset:]
    x = wide.view(b, L, 2 * d)[..., :d].transpose(1, 2)
    w = torch.randn(d, 4, device="cuda", generator=gen)
    for bias in (torch.randn(d, device="cuda", generator=gen), None):
        y = arm.causal_conv1d(x, w, bias, activation=act, time_major=True)
        assert y.transpose(1, 2).is_contiguous()
        assert torch.equal(y, arm.causal_conv1d(x, w, bias, activation=act))
