"""selective_scan_time_major on rows of any length, B and C as a projection's columns:
the bits of the contiguous scan of the same values (whose parity with the oracle is
test_m1_gpu.py's), at lengths around the chunk of 256 steps and the packing's 64."""

import pytest

from util import case

pytestmark = pytest.mark.gpu

SHAPES = [
    # (batch, dim, len, state, groups)
    (1, 16, 1, 16, 1),
    (2, 48, 77, 16, 1),
    (1, 32, 63, 13, 2),
    (2, 64, 257, 16, 2),
    (1, 32, 1531, 16, 1),    # few rows: segments, whose fold reads u by strides
    (3, 16, 2047, 17, 1),
    (8, 1024, 301, 16, 1),   # whole rows
    (1, 32, 1026, 16, 1),
]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("reverse", [False, True])
def test_views_equal_contiguous(shape, reverse):
    import torch

    import armhackathon_amd as arm
    from armhackathon_amd import op

    b, d, L, n, g = shape
    gen = torch.Generator(device="cuda").manual_seed(L + n)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=gen)  # noqa: E731
    x, z = rnd(b, L, 2 * d).transpose(1, 2).chunk(2, dim=1)
    delta = rnd(b, d, L) * 0.5 - 3
    A, D, bias, h0 = -torch.rand(d, n, device="cuda") * 4, rnd(d), rnd(d), rnd(b, d, n)
    cols = rnd(b, L, 20 + 2 * g * n)
    B = cols[..., 20:20 + g * n].unflatten(-1, (g, n)).permute(0, 2, 3, 1)
    C = cols[..., 20 + g * n:].unflatten(-1, (g, n)).permute(0, 2, 3, 1)
    for u, zz, h, cc in ((x, z, None, C), (x.contiguous(), z, h0, C.contiguous()),
                         (x, None, h0, C)):
        case(f"views {shape} reverse={reverse} u {u.stride()} z={zz is not None}")
        kw = dict(D=D, delta_bias=bias, delta_softplus=True, return_last_state=True,
                  initial_state=h, reverse=reverse)
        assert op.front().selective_scan_time_major(u, delta, A, B, cc, D, zz, bias, h, True,
                                                    reverse) is not None  # served in place
        out, last = arm.selective_scan_time_major(u, delta, A, B, cc, z=zz, **kw)
        want, wlast = arm.selective_scan(u.contiguous(), delta, A, B.contiguous(),
                                         cc.contiguous(),
                                         z=None if zz is None else zz.contiguous(), **kw)
        assert out.transpose(1, 2).is_contiguous()
        assert torch.equal(out, want) and torch.equal(last, wlast)


def test_views_left_to_the_copy():
    """Few states with odd rows, and a dim off the 16-row blocks: the copying route."""
    import torch

    import armhackathon_amd as arm
    from armhackathon_amd import op

    for d, n, L in ((32, 8, 77), (24, 16, 64)):
        case(f"not served in place: dim {d} state {n} len {L}")
        z, dl, B = (torch.randn(*s, device="cuda") for s in ((1, L, d), (1, d, L), (1, n, L)))
        A, z = -torch.rand(d, n, device="cuda"), z.transpose(1, 2)
        assert op.front().selective_scan_time_major(z, dl, A, B, B, None, z, None, None, True,
                                                    False) is None
        assert torch.equal(
            arm.selective_scan_time_major(z, dl, A, B, B, z=z, delta_softplus=True),
            arm.selective_scan(z, dl, A, B, B, z=z, delta_softplus=True))
