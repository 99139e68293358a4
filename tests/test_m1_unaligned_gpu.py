"""Rows that are not 16-byte multiples through the tiled kernel, at the lengths where a
16-byte load meets a row's end: rows shorter than a piece, a piece or a lane block crossing
the end, one step around a chunk, whole rows and segments, against float64.

Gate 2e-6 of the largest value: sums of 16 products of states that decay (16 * 2^-24 = 1e-6
at worst). A step read from a neighbouring row or a shifted piece is off by its whole value.
"""

import numpy as np
import pytest

from oracle import naive
from util import case, host, rel_err

pytestmark = pytest.mark.gpu


LENGTHS = [1, 2, 3, 5, 6, 7, 17, 18, 19, 31, 253, 254, 255, 257, 259, 511, 769, 1538]


def _inputs(length):
    import torch

    rng = np.random.default_rng(length)
    b, d, n = 2, 32, 16
    f = lambda *s: rng.standard_normal(s).astype(np.float32)  # noqa: E731
    x = dict(u=f(b, d, length), delta=f(b, d, length) * 0.5 - 3, A=-np.exp(f(d, n)),
             B=f(b, n, length), C=f(b, n, length), D=f(d), z=f(b, d, length), bias=f(d))
    t = {k: torch.from_numpy(np.ascontiguousarray(v)).cuda() for k, v in x.items()}
    kw = dict(D=t["D"], z=t["z"], delta_bias=t["bias"], delta_softplus=True)
    return x, [t[k] for k in ("u", "delta", "A", "B", "C")], kw


def _want(x, reverse):
    return naive.m1_scan(x["u"], x["delta"], x["A"], x["B"], x["C"], D=x["D"], z=x["z"],
                         delta_bias=x["bias"], delta_softplus=True, reverse=reverse)


@pytest.mark.parametrize("length", LENGTHS)
@pytest.mark.parametrize("reverse", [False, True])
def test_row_ends(length, reverse):
    import armhackathon_amd as arm

    case(f"unaligned rows L {length} reverse={reverse}")
    x, args, kw = _inputs(length)
    want, last = _want(x, reverse)
    out, got = arm.selective_scan(*args, reverse=reverse, return_last_state=True, **kw)
    assert rel_err(host(got), last) < 2e-6
    assert rel_err(host(out), want) < 2e-6


@pytest.mark.parametrize("length", LENGTHS)
def test_row_ends_of_a_pair(length):
    """Both directions in one launch."""
    import armhackathon_amd as arm

    case(f"unaligned rows L {length}, both directions")
    x, args, kw = _inputs(length)
    for out, reverse in zip(arm.bidirectional_scan(*args, merge="none", **kw), (False, True)):
        assert rel_err(host(out), _want(x, reverse)[0]) < 2e-6
