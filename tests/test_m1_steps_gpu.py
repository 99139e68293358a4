"""The decode steps' 16-byte kernels at the edges of their ranges, against float64: states
of 1 to 16 lanes a row, blocks whose last rows are missing, B and C by pieces or by strides,
a window of another width or alignment (the one-thread kernels).

Gate 2e-6 of the sum of the absolute terms of the largest output, which is what bounds the
rounding of a 32-bit sum whose terms cancel (a single row's y may be small beside them): up
to 144 products and roundings of 2^-24 each (8.6e-6 at worst, their square root, 7e-7,
typical) of states that one 32-bit exponential and two roundings make.
"""

import pytest

from util import case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4, 8, 12, 16, 64, 128, 144, 6])
@pytest.mark.parametrize("rows", [(1, 1), (3, 37), (40, 1536)], ids=lambda r: "%dx%d" % r)
@pytest.mark.parametrize("columns", [False, True])
def test_state_update(n, rows, columns):
    import torch

    import armhackathon_amd as arm

    b, d = rows
    case(f"state update {b}x{d} N {n} columns={columns}")
    gen = torch.Generator(device="cuda").manual_seed(n + d)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=gen)  # noqa: E731
    x, dt, z, A = rnd(b, d), rnd(b, d) - 3, rnd(b, d), -torch.exp(rnd(d, n))
    wide = rnd(b, 2 * n + 4)
    B, C = ((wide[:, 4:4 + n], wide[:, 4 + n:]) if columns
            else (rnd(b, n + 1)[:, 1:], rnd(n, b).t()))
    D, bias, h = rnd(d), rnd(d), rnd(b, d, n)
    f = lambda t: t.double()  # noqa: E731
    dt64 = torch.nn.functional.softplus(f(dt) + f(bias))
    want_h = torch.exp(dt64[..., None] * f(A)) * f(h) + (dt64 * f(x))[..., None] * f(B)[:, None]
    want = ((want_h * f(C)[:, None]).sum(-1) + f(D) * f(x)) * torch.nn.functional.silu(f(z))
    terms_h = (torch.exp(dt64[..., None] * f(A)) * f(h)).abs() \
        + ((dt64 * f(x))[..., None] * f(B)[:, None]).abs()
    terms = ((terms_h * f(C)[:, None].abs()).sum(-1) + (f(D) * f(x)).abs()) \
        * torch.nn.functional.silu(f(z)).abs()
    y = arm.selective_state_update(h, x, dt, A, B, C, D=D, z=z, dt_bias=bias, dt_softplus=True)
    for got, ref, scale in ((y, want, terms), (h, want_h, terms_h)):
        assert ((got.double() - ref).abs().max() / scale.max()).item() < 2e-6


@pytest.mark.parametrize("width,offset", [(4, 0), (4, 1), (3, 0), (8, 0)])
@pytest.mark.parametrize("rows", [(1, 1), (3, 37), (48, 1536)], ids=lambda r: "%dx%d" % r)
def test_conv_step(width, offset, rows):
    import torch

    import armhackathon_amd as arm

    b, d = rows
    case(f"conv step {b}x{d} width {width} offset {offset}")
    gen = torch.Generator(device="cuda").manual_seed(width + d)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=gen)  # noqa: E731
    s = rnd(b * d * width + offset)[offset:].view(b, d, width)
    w, bias, x = rnd(d, width), rnd(d), rnd(b, 2 * d)[:, d:]
    win = torch.cat((s[..., 1:], x[..., None]), -1)
    want = torch.nn.functional.silu((win.double() * w.double()).sum(-1) + bias.double())
    y = arm.causal_conv1d_update(x, s, w, bias, activation="silu")
    assert torch.equal(s, win)
    terms = (win.double() * w.double()).abs().sum(-1) + bias.double().abs()
    assert ((y.double() - want).abs().max() / terms.max()).item() < 2e-6
