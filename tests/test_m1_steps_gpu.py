"""The decode steps' 16-byte kernels at the edges of their ranges, against float64: states
of 1 to 16 lanes a row, blocks whose last rows are missing, B and C by pieces or by strides,
a window of another width or alignment (the one-thread kernels).

Every element is held to the bound of its own roundings, in units e = 2^-24 of its terms'
absolute values (an output may be small beside terms that cancel):
- dt = softplus(s): s rounded (|s| e), exp by exp2 of a rounded argument (2 |s| e, and 2 e for
  exp2's own ulp), log1p 6 e: (3 |s| + 8) e;
- exp(dt A): the relative error of dt and three roundings of the argument, times |dt A|, and
  2 e; the state two more: (3 |s| + 12) e of e^{dt A} |h| (1 + |dt A|) + |dt x B|;
- y: the states' errors and up to 45 e of sums (144 states on four lanes), silu (2 |z| + 6) e.
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
    decayed = (torch.exp(dt64[..., None] * f(A)) * f(h)).abs()
    inflow = ((dt64 * f(x))[..., None] * f(B)[:, None]).abs()
    err_h = (3 * (f(dt) + f(bias)).abs() + 12)[..., None] \
        * (decayed * (1 + (dt64[..., None] * f(A)).abs()) + inflow)
    silu = torch.nn.functional.silu(f(z)).abs()
    terms = (decayed + inflow) * f(C)[:, None].abs()
    skip = (f(D) * f(x)).abs()
    err_y = silu * ((err_h * f(C)[:, None].abs()).sum(-1) + 45 * (terms.sum(-1) + skip)
                    + (2 * f(z).abs() + 6) * (terms.sum(-1) + skip))
    y = arm.selective_state_update(h, x, dt, A, B, C, D=D, z=z, dt_bias=bias, dt_softplus=True)
    for got, ref, err in ((y, want, err_y), (h, want_h, err_h)):
        assert ((got.double() - ref).abs() / err).max().item() < 2.0 ** -24


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
    # the sum (a rounding a tap), through silu's slope of at most 1.1, and silu itself
    acc = (win.double() * w.double()).sum(-1) + bias.double()
    terms = (win.double() * w.double()).abs().sum(-1) + bias.double().abs()
    err = 1.1 * (width + 1) * terms + (2 * acc.abs() + 6) * want.abs()
    assert ((y.double() - want).abs() / err).max().item() < 2.0 ** -24
