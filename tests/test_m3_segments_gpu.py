"""Mamba-3 sequences cut into equal segments (few sequences for the chip: several
resuming blocks per sequence, each starting from the fold pieces before it), against the
float64 oracle: outputs, final states and last_bx, at the lengths where the plan changes.

Gate 1e-5 of the tensor's largest value: the products are 32-bit sums of up to 128 terms
(128 * 2^-24 = 7.6e-6 at worst, 2^-24 sqrt(128) = 7e-7 typical), and a piece combined in
the wrong order, twice or not at all changes the state by its whole share.
"""

import numpy as np
import pytest

import oracle
from armhackathon_amd import workloads
from util import case, dev, host, rel_err

pytestmark = pytest.mark.gpu

TOL = 1e-5
KEYS = ("q", "k", "v", "adt", "dt", "trap", "q_bias", "k_bias")


def _inputs(rank, b, L, h, dv, dqk, g):
    x = (workloads.m3_mimo(batch=b, length=L, heads=h, dv=dv, dqk=dqk, rank=rank, seed=L)
         if rank else workloads.m3_siso(batch=b, length=L, heads=h, dv=dv, dqk=dqk, seed=L))
    x["q"], x["k"] = (np.ascontiguousarray(x[n][..., :g, :]) for n in ("q", "k"))
    rng = np.random.default_rng(L + 1)
    for n in ("q_bias", "k_bias"):
        x[n] = (rng.standard_normal(x[n].shape) * 0.1).astype(np.float32)
    x["D"] = rng.standard_normal(h).astype(np.float32)
    x["z"] = rng.standard_normal(x["v"].shape).astype(np.float32)
    if rank:
        x["zeta"] = rng.standard_normal(x["zeta"].shape).astype(np.float32)
    return x


CASES = [
    # (rank or 0 for SISO, batch, length, heads, dv, dqk, groups)
    (0, 1, 368, 3, 64, 128, 1),    # 23 chunks: whole
    (0, 1, 369, 3, 64, 128, 3),    # 24, the last of one step: the shortest cut
    (0, 1, 1033, 1, 32, 128, 1),   # 13 segments of five chunks, one block each
    (0, 1, 3000, 1, 32, 128, 1),   # 47 segments, more pieces than a segment's cap, one XCD
    (0, 1, 2304, 12, 32, 64, 1),   # 12 sequences: uneven over the XCDs, in several rounds
    (0, 2, 900, 24, 64, 128, 1),   # 96 blocks: two segments
    (0, 1, 1500, 24, 64, 64, 1),   # 48 blocks: segments rounded up to whole pieces
    (2, 1, 261, 5, 64, 128, 5),
    (4, 1, 93, 3, 64, 128, 1),     # 24 chunks of four steps
    (4, 2, 530, 8, 64, 64, 1),
    (4, 1, 1100, 1, 32, 64, 1),    # 275 chunks: 55 segments
]


@pytest.mark.parametrize("shape", CASES, ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("reverse", [False, True])
def test_m3_equal_segments(shape, reverse):
    import armhackathon_amd as arm_scan

    case(f"equal segments {shape} reverse={reverse}")
    rank, L = shape[0], shape[2]
    x = _inputs(*shape)
    kw = dict(psi=x["psi"], zeta=x["zeta"], phi=x["phi"]) if rank else {}
    ref, rls, rbx = oracle.mamba3_scan(*[x[k] for k in KEYS], x["cos"], x["sin"], D=x["D"],
                                       z=x["z"], reverse=reverse, want_state=True,
                                       dtype=np.float64, **kw)
    t = dev(x)
    args = [t[k] for k in KEYS]
    if rank:
        out, ls = arm_scan.mamba3_mimo_scan(*args, t["psi"], t["zeta"], t["phi"], cos=t["cos"],
                                            sin=t["sin"], D=t["D"], z=t["z"], reverse=reverse,
                                            return_last_state=True)
    else:
        out, ls, bx = arm_scan.mamba3_scan(*args, cos=t["cos"], sin=t["sin"], D=t["D"],
                                           z=t["z"], reverse=reverse, return_last_state=True)
        assert rel_err(host(bx), rbx) < TOL
    assert out.shape[1] == L
    assert rel_err(host(out), ref.transpose(0, 2, 1, 3)) < TOL
    assert rel_err(host(ls), rls) < TOL


@pytest.mark.parametrize("shape", [c for c in CASES if not c[0]],
                         ids=lambda c: "x".join(map(str, c)))
def test_m3_equal_segments_fused_angles(shape):
    """Raw angles: each piece rotates from its own start, the resuming blocks by the
    angles summed before it."""
    import armhackathon_amd as arm_scan

    case(f"equal segments, fused angles {shape}")
    x = _inputs(*shape)
    x = workloads.m3_with_angles(x, seed=3)
    cos, sin = oracle.angles_to_cos_sin(x["angles"].astype(np.float64),
                                        x["dt"].astype(np.float64), x["q"].shape[-1] // 2)
    ref, rls, rbx = oracle.mamba3_scan(*[x[k] for k in KEYS], cos, sin, D=x["D"], z=x["z"],
                                       want_state=True, dtype=np.float64)
    t = dev(x)
    out, ls, bx = arm_scan.mamba3_scan(*[t[k] for k in KEYS], angles=t["angles"], D=t["D"],
                                       z=t["z"], return_last_state=True)
    for got, want in ((out, ref.transpose(0, 2, 1, 3)), (ls, rls), (bx, rbx)):
        assert rel_err(host(got), want) < TOL


def test_m3_equal_segments_noncausal():
    """The accumulating backward traversal on equal segments equals forward + backward
    without the same-step term counted twice."""
    import armhackathon_amd as arm_scan
    from oracle import naive

    case("equal segments, non-causal")
    x = _inputs(0, 1, 777, 3, 64, 128, 1)
    args = [x[k] for k in KEYS] + [x["cos"], x["sin"]]
    both = [oracle.mamba3_scan(*args, D=x["D"], z=x["z"], reverse=r, dtype=np.float64)
            for r in (False, True)]
    ref = sum(y.transpose(0, 2, 1, 3) for y in both) - naive.m3_same_step(
        x["q"], x["k"], x["v"], x["dt"], x["trap"], x["q_bias"], x["k_bias"], D=x["D"],
        z=x["z"])
    t = dev(x)
    out = arm_scan.noncausal_scan(*[t[k] for k in KEYS], cos=t["cos"], sin=t["sin"], D=t["D"],
                                  z=t["z"])
    assert rel_err(host(out), ref) < TOL
