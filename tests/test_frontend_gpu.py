"""The mixer's front-end kernel where its norm rows move by 16-byte pieces (row stride and
bases multiples of 4 floats) and where they do not, at rows of 1 to 64 lanes and more, and
token counts that leave gate and norm blocks partly empty, against float64.

Gate 4e-6 of the largest value: a sum of up to 320 squares (320 * 2^-24 = 1.9e-5 at worst,
halved by the square root, its own square root typical), two divisions and two products.
"""

import numpy as np
import pytest

from oracle import naive
from util import case, host, rel_err

pytestmark = pytest.mark.gpu

TOL = 4e-6


@pytest.mark.parametrize("n", [4, 32, 64, 128, 256, 260, 320, 30])
@pytest.mark.parametrize("tokens", [(1, 1), (2, 33), (1, 257)], ids=lambda t: "%dx%d" % t)
@pytest.mark.parametrize("aligned", [True, False])
def test_rows(n, tokens, aligned):
    import torch

    from armhackathon_amd import _ffi

    (b, L), h, hd, rank, groups, nang = tokens, 3, 16, 2, 1, 4
    case(f"front-end n {n} tokens {b}x{L} aligned={aligned}")
    bc = rank * groups * n
    need = 2 * h * hd + 2 * bc + 3 * h + nang
    rs = (need + 3) // 4 * 4 + (0 if aligned else 1)
    rng = np.random.default_rng(n + L)
    proj = rng.standard_normal((b, L, rs)).astype(np.float32)
    bias = rng.uniform(-4, -2, h).astype(np.float32)
    wb, wc = (1 + 0.3 * rng.standard_normal((2, n))).astype(np.float32)
    t = [torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in (proj, bias, wb, wc)]
    q = torch.full((b, L, rank, groups, n), float("nan"), device="cuda")
    k = q.clone()
    adt, dt, trap = torch.full((3, b, h, L), float("nan"), device="cuda").unbind(0)
    _ffi.block_frontend_raw(t[0].data_ptr(), b, L, rs, h, hd, n, rank, groups, nang,
                            t[1].data_ptr(), 1e-4, t[2].data_ptr(), t[3].data_ptr(), 1e-5,
                            q.data_ptr(), k.data_ptr(), adt.data_ptr(), dt.data_ptr(),
                            trap.data_ptr())
    torch.cuda.synchronize()
    p = proj.astype(np.float64)
    o = 2 * h * hd
    B, C = (p[..., s:s + bc].reshape(b, L, rank, groups, n) for s in (o, o + bc))
    g = p[..., o + 2 * bc:]
    DT = naive.softplus(g[..., :h] + bias)
    ADT = np.minimum(-naive.heavy_tail(g[..., h:2 * h]), -1e-4) * DT
    for got, want in ((k, naive.rms_norm(B, wb, 1e-5)), (q, naive.rms_norm(C, wc, 1e-5)),
                      (dt, DT.transpose(0, 2, 1)), (adt, ADT.transpose(0, 2, 1)),
                      (trap, g[..., 2 * h:3 * h].transpose(0, 2, 1))):
        assert rel_err(host(got), want) <= TOL
