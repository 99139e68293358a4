"""The native eager front-end (csrc/torch_front.cpp): a plain call has the bits of the
custom op's, and whatever is not plain is left to the custom op, which records, refuses or
raises as it did."""

import pytest

from util import case

pytestmark = pytest.mark.gpu


def _rand(*shape, seed=0, scale=1.0):
    import torch

    g = torch.Generator(device="cuda").manual_seed(seed + sum(shape))
    return torch.randn(*shape, device="cuda", generator=g) * scale


def _calls():
    import torch
    import torch.nn.functional as F

    import armhackathon_amd as arm
    from armhackathon_amd.mamba3_block import Mamba3Mixer

    b, d, n, L = 2, 32, 16, 260
    u, dl = _rand(b, d, L), _rand(b, d, L, seed=1) - 3
    A, D, bias = -torch.rand(d, n, device="cuda"), _rand(d, seed=2), _rand(d, seed=3)
    B, C, z = _rand(b, n, L, seed=4), _rand(b, n, L, seed=5), _rand(b, d, L, seed=6)
    Bs = _rand(b, L, 40, seed=7)[..., 8:8 + n].transpose(1, 2)  # a projection's columns
    tm = _rand(b, L, 2 * d, seed=8).transpose(1, 2)
    h0 = _rand(b, d, n, seed=9)
    kw = dict(D=D, z=z, delta_bias=bias, delta_softplus=True)
    w, wb = _rand(d, 4, seed=10), _rand(d, seed=11)
    calls = {
        "scan": lambda: arm.selective_scan(u, dl, A, B, C, return_last_state=True,
                                           initial_state=h0, **kw),
        "scan_reverse_groups": lambda: arm.selective_scan(
            u, dl, A, B.view(b, 1, n, L).repeat(1, 2, 1, 1), C.view(b, 1, n, L).repeat(1, 2, 1, 1),
            reverse=True, delta_softplus=True),
        "scan_views": lambda: arm.selective_scan(tm[:, :d], dl, A, Bs, C, z=tm[:, d:],
                                                 delta_softplus=True),
        "time_major": lambda: arm.selective_scan_time_major(
            tm[:, :d], dl, A, Bs, C, D=D, z=tm[:, d:], delta_softplus=True,
            return_last_state=True),
        "bidir": lambda: arm.bidirectional_scan(u, dl, A, B, C, merge="none", **kw),
        "conv": lambda: arm.causal_conv1d(tm[:, :d], w, wb, activation="silu", time_major=True),
        "conv_plain": lambda: arm.causal_conv1d(u, w),
    }

    def steps():
        cs, hs = _rand(b, d, 4, seed=12), _rand(b, d, n, seed=13)
        x = arm.causal_conv1d_update(tm[:, :d, 3], cs, w, wb, activation="silu")
        y = arm.selective_state_update(hs, x, dl[..., 0], A, Bs[..., 0], C[..., 0], D=D,
                                       z=z[..., 0], dt_bias=bias, dt_softplus=True)
        return x, y, cs, hs

    calls["steps"] = steps
    H = 7
    grid = [_rand(b, d, H, H, seed=s) for s in (20, 21, 22)]
    B4, C4 = _rand(4, b, n, H, H, seed=23), _rand(4, b, n, H, H, seed=24)
    calls["ss2d"] = lambda: arm.ss2d_scan(grid[0], grid[1] - 3, A, B4, C4, D=D, z=grid[2],
                                          per_direction=True, return_last_state=True)
    calls["ss2d_none"] = lambda: arm.ss2d_scan(grid[0], grid[1] - 3, A, B4[0], C4[0],
                                               merge="none")
    h, dv, dqk, Lm = 4, 32, 64, 75
    dt = F.softplus(_rand(b, h, Lm, seed=30) - 3)
    args = [_rand(b, Lm, dqk, seed=31, scale=0.1), _rand(b, Lm, 1, dqk, seed=32, scale=0.1),
            _rand(b, Lm, h, dv, seed=33), -0.5 * dt, dt, _rand(b, h, Lm, seed=34),
            _rand(h, dqk, seed=35, scale=0.1), _rand(h, dqk, seed=36, scale=0.1)]
    ang, zz, Dh = _rand(b, Lm, h, 16, seed=37), _rand(b, Lm, h, dv, seed=38), _rand(h, seed=39)
    cos, sin = arm.angles_to_cos_sin(ang, dt, dqk // 2)
    shared = _rand(b, Lm, 1, 16, seed=40).expand(b, Lm, h, 16)
    odd = _rand(b * Lm * h * 16 + 1, seed=41)[1:].view(b, Lm, h, 16)  # off a 16-byte base
    for name, kw3 in dict(cos=dict(cos=cos, sin=sin), cos_reverse=dict(cos=cos, sin=sin,
                                                                       reverse=True),
                          angles=dict(angles=ang), angles_reverse=dict(angles=ang, reverse=True),
                          angles_shared=dict(angles=shared), angles_odd=dict(angles=odd),
                          carry=dict(angles=ang, return_last_state=True)).items():
        calls["m3_" + name] = lambda kw3=kw3: arm.mamba3_scan(*args, D=Dh, z=zz, **kw3)
    m = list(args)
    m[0], m[1] = _rand(b, Lm, 4, dqk, seed=42), _rand(b, Lm, 4, 2, dqk, seed=43)
    m[0] = m[0].unsqueeze(3).repeat(1, 1, 1, 2, 1)
    m[6], m[7] = _rand(h, 4, dqk, seed=44), _rand(h, 4, dqk, seed=45)
    ranks = [_rand(h, 4, dv, seed=s) for s in (46, 47, 48)]
    for name, kw3 in dict(cos=dict(cos=cos, sin=sin, return_last_state=True),
                          angles=dict(angles=ang), shared=dict(angles=shared),
                          reverse=dict(angles=ang, reverse=True)).items():
        calls["mimo_" + name] = lambda kw3=kw3: arm.mamba3_mimo_scan(*m, *ranks, D=Dh, z=zz,
                                                                     **kw3)
    calls["noncausal"] = lambda: arm.noncausal_scan(*args, angles=ang, D=Dh, z=zz)
    mixer = Mamba3Mixer(d_model=64, d_state=32, headdim=32).to("cuda").requires_grad_(False)
    x = _rand(b, Lm, 64, seed=50)
    calls["mixer"] = lambda: mixer(x)
    return calls


def test_same_bits_as_the_custom_op(monkeypatch):
    import torch

    from armhackathon_amd import op

    flat = lambda r: list(r) if isinstance(r, tuple) else [r]  # noqa: E731
    leaves = lambda r: [t for x in flat(r) for t in flat(x)]  # noqa: E731
    served, calls = [], _calls()
    real = op.front()  # the GPU is in use from here on
    for name, call in calls.items():
        case(f"front-end {name}")

        class Spy:
            def __getattr__(self, fn):
                def run(*a):
                    r = getattr(real, fn)(*a)
                    served.append((name, fn, r is not None))
                    return r
                return run

        monkeypatch.setattr(op, "front", lambda: Spy())
        got = leaves(call())
        monkeypatch.setattr(op, "front", lambda: None)
        want = leaves(call())
        assert len(got) == len(want)
        for g, w in zip(got, want):
            assert g.shape == w.shape and g.stride() == w.stride() and torch.equal(g, w), name
    assert served and all(ok for _, _, ok in served), [s for s in served if not s[2]]


def test_not_plain_is_left_alone():
    import torch
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    import armhackathon_amd as arm
    from armhackathon_amd import op

    b, d, n, L = 1, 16, 8, 40
    u, dl = _rand(b, d, L), _rand(b, d, L, seed=1)
    A, B = -torch.rand(d, n, device="cuda"), _rand(b, n, L, seed=2)
    f = op.front()

    def native(u=u, dl=dl):
        return f.selective_scan(u, dl, A, B, B, None, None, None, None, True, False)

    assert native() is not None
    for bad in (u.double(), u.cpu(), u[0], u[:, :, :0], u.clone().requires_grad_(), None, 3,
                torch.nn.Parameter(u.clone())):
        case(f"not plain: {type(bad).__name__}")
        assert native(u=bad) is None
    assert native(dl=dl[..., :-1]) is None
    with torch.no_grad():
        assert native(u=u.clone().requires_grad_()) is not None
    with torch.inference_mode():
        assert native() is not None

    class Fn(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Disp(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    for mode in (Fn(), Disp()):
        with mode:
            assert native() is None
    seen = []

    def inner(x):
        seen.append(native(u=x) is None)
        return x

    torch.vmap(inner)(u.unsqueeze(0))
    with torch.autograd.forward_ad.dual_level():
        seen.append(native(u=torch.autograd.forward_ad.make_dual(u, u)) is None)
    assert seen == [True, True]
    with pytest.raises(ValueError):
        arm.selective_scan(u, dl[..., :-1], A, B, B)
    y = arm.selective_scan(u.clone().requires_grad_(), dl, A, B, B, delta_softplus=True)
    with pytest.raises(RuntimeError):
        y.sum().backward()


def test_state_version_counts():
    """The states written in place count as written, as an op that mutates them does."""
    import torch

    import armhackathon_amd as arm

    s, x = torch.zeros(1, 16, 4, device="cuda"), _rand(1, 16)
    before = s._version
    arm.causal_conv1d_update(x, s, _rand(16, 4, seed=1))
    assert s._version > before
    h = torch.zeros(1, 16, 8, device="cuda")
    before = h._version
    arm.selective_state_update(h, x, x, -torch.rand(16, 8, device="cuda"), _rand(1, 8), _rand(1, 8))
    assert h._version > before


def test_scratch_during_capture():
    """Captured with torch's graphs, a call takes its scratch from the graph's own blocks of
    torch's allocator; each replay equals the eager result, with eager calls between that
    reuse torch's other blocks."""
    import torch

    import armhackathon_amd as arm

    b, d, n, L = 1, 32, 16, 1024  # few rows: the segment maps are scratch
    u, dl = _rand(b, d, L), _rand(b, d, L, seed=1)
    A, B = -torch.rand(d, n, device="cuda"), _rand(b, n, L, seed=2)
    run = lambda: arm.selective_scan(u, dl, A, B, B, delta_softplus=True)  # noqa: E731
    want = run().clone()
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(st):
        run()
    torch.cuda.current_stream().wait_stream(st)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = run()
    for i in range(4):
        case(f"replay {i}")
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        torch.full((4096, 256), float(i), device="cuda")
        assert torch.equal(run(), want)


@pytest.mark.parametrize("native", [True, False], ids=["front-end", "custom op"])
def test_autocast_changes_nothing(native, monkeypatch):
    """The ops have no autocast rule: a float32 call is the same under it, on either route."""
    import torch

    from armhackathon_amd import op

    if not native:
        monkeypatch.setattr(op, "front", lambda: None)
    calls = _calls()
    for name in ("scan_views", "bidir", "m3_cos"):
        case(f"autocast, {'front-end' if native else 'custom op'}: {name}")
        want = calls[name]()
        with torch.autocast("cuda", dtype=torch.bfloat16):
            got = calls[name]()
        flat = lambda r: r if isinstance(r, tuple) else (r,)  # noqa: E731
        for g, w in zip(flat(got), flat(want)):
            assert g.dtype == torch.float32 and torch.equal(g, w)


def _allocations():
    import torch

    return torch.cuda.memory_stats()["allocation.all.allocated"]


def test_refusals_allocate_nothing():
    """What is left to the custom op has been copied and allocated by nobody yet."""
    import torch

    from armhackathon_amd import op

    f, no = op.front(), (None,) * 4
    b, d, n, L = 2, 32, 16, 77
    u, A, B = _rand(b, d, L), -torch.rand(n, d, device="cuda").t(), _rand(b, L, n).transpose(1, 2)
    tm = _rand(b, L, d).transpose(1, 2)  # as delta: a copy where it is taken
    few, B8 = -torch.rand(d, 8, device="cuda"), _rand(b, 8, L)
    grid, B4 = _rand(b, d, 7, 7), _rand(4, b, n, 7, 7)
    q, v, g = _rand(b, 64, L).transpose(1, 2), _rand(b, L, 4, 32), _rand(b, 4, L)
    bias, cos = _rand(4, 64), _rand(b, L, 4, 32)
    wants_grad, state = torch.nn.Parameter(bias.clone()), torch.zeros(b, d, n, device="cuda")
    refused = {
        "dim 24": lambda: f.selective_scan_time_major(tm[:, :24], tm[:, :24], A[:24], B, B, *no,
                                                      True, False),
        "8 states, odd rows": lambda: f.selective_scan_time_major(
            tm, tm, few, B8, B8, None, tm, None, None, True, False),
        "z not by channels": lambda: f.selective_scan_time_major(tm, tm, A, B, B, None, u, None,
                                                                 None, True, False),
        "scan, h0 of another shape": lambda: f.selective_scan(tm, tm, A, B, B, None, tm, None,
                                                              u, True, False),
        "ss2d, z of another shape": lambda: f.ss2d(grid.transpose(2, 3), grid, A, B4, B4, None,
                                                   u, None, True, 1, False),
        "mamba3, a gradient": lambda: f.mamba3(q, q, v, g, g, g, bias, wants_grad, cos, cos, None,
                                               *no, None, False, False, False),
        "step, z of another shape": lambda: f.state_update(
            state, u[..., 0], u[..., 1], A, B[..., 0], B[..., 0], None, u, None, True),
    }
    for name, call in refused.items():
        case(f"refused: {name}")
        before = _allocations()
        assert call() is None
        assert _allocations() == before, name


def test_views_rule_is_the_library_s():
    """The front-end takes a time-major call where the library's views entry does."""
    import ctypes
    import itertools

    import torch

    from armhackathon_amd import _ffi, op

    f, lib, b, d = op.front(), _ffi.load(), 2, 32

    def strides(t, k):
        return (ctypes.c_longlong * k)(*t.stride())

    def layouts(L):
        wide = _rand(b, L, 2 * d + 4, seed=L)
        flat = _rand(b * d * L + 1, seed=L + 1)
        return {"rows": _rand(b, d, L), "rows, off 16 bytes": flat[1:].view(b, d, L),
                "columns": wide[..., :d].transpose(1, 2),
                "columns, off 16 bytes": wide[..., 1:1 + d].transpose(1, 2),
                "columns, odd steps": _rand(b, L, d + 1)[..., :d].transpose(1, 2)}

    taken = set()
    for L, n in itertools.product((1, 64, 77), (8, 16)):
        A, B = -torch.rand(d, n, device="cuda"), _rand(b, 1, n, L)
        x = layouts(L)
        for un, zn, dn in itertools.product(x, [None, *x], ("rows", "rows, off 16 bytes")):
            case(f"views L {L} states {n}: u {un}, z {zn}, delta {dn}")
            u, delta, z = x[un], x[dn], None if zn is None else x[zn]
            got = f.selective_scan_time_major(u, delta, A, B, B, None, z, None, None, True, False)
            out = torch.empty(b, L, d, device="cuda").transpose(1, 2)
            rc = lib.arm_scan_selective_scan_views_f32(
                ctypes.byref(_ffi.ArmScanDims(b, d, L, n, 1)), u.data_ptr(),
                None if u.is_contiguous() else strides(u, 3), delta.data_ptr(), A.data_ptr(),
                B.data_ptr(), strides(B, 4), B.data_ptr(), strides(B, 4), None,
                None if z is None else z.data_ptr(), None if z is None else strides(z, 3), None,
                1, 0, out.data_ptr(), strides(out, 3), None, None,
                torch.cuda.current_stream().cuda_stream)
            assert rc in (0, 2) and (got is None) == (rc == 2)
            if rc == 0:
                assert torch.equal(got[0], out)
            taken.add(rc)
    assert taken == {0, 2}


def _node_types(graph):
    import ctypes

    hip = ctypes.CDLL("libamdhip64.so.7")
    vp = ctypes.c_void_p
    hip.hipGraphGetNodes.argtypes = [vp, vp, ctypes.POINTER(ctypes.c_size_t)]
    hip.hipGraphNodeGetType.argtypes = [vp, ctypes.POINTER(ctypes.c_int)]
    count = ctypes.c_size_t(0)
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(count)) == 0
    nodes = (vp * max(count.value, 1))()
    assert hip.hipGraphGetNodes(graph, nodes, ctypes.byref(count)) == 0
    kinds = set()
    for i in range(count.value):
        kind = ctypes.c_int(-1)
        assert hip.hipGraphNodeGetType(nodes[i], ctypes.byref(kind)) == 0
        kinds.add(kind.value)
    return kinds


@pytest.mark.parametrize("native", [True, False], ids=["front-end", "custom op"])
def test_capture_records_kernels_only(native, monkeypatch):
    """No call leaves an allocation or a free in a captured graph, whichever way it goes: its
    scratch is torch's. The graphs are looked at and not launched."""
    import torch

    from armhackathon_amd import op

    calls = _calls()
    names = ("m3_cos", "m3_angles_odd", "m3_carry", "mimo_angles", "ss2d", "noncausal", "bidir",
             "scan_views")
    for name in names:
        calls[name]()
    if not native:
        monkeypatch.setattr(op, "front", lambda: None)
    for name in names:
        case(f"capture, {'front-end' if native else 'custom op'}: {name}")
        g = torch.cuda.CUDAGraph(keep_graph=True)
        with torch.cuda.graph(g):
            out = calls[name]()
        assert _node_types(g.raw_cuda_graph()) == {0}, name  # hipGraphNodeTypeKernel
        del out, g


def test_capture_without_a_source_of_scratch_is_refused():
    """Through the C ABI alone a captured call that needs scratch fails, and nothing of it is
    recorded."""
    import ctypes

    import torch

    from armhackathon_amd import _ffi

    b, d, n, L = 1, 32, 16, 1024
    u, dl = _rand(b, d, L), _rand(b, d, L, seed=1)
    A, B, out = -torch.rand(d, n, device="cuda"), _rand(b, n, L, seed=2), torch.empty_like(u)
    case("capture through the C ABI")
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(g):
        rc = _ffi.load().arm_scan_selective_scan_f32(
            ctypes.byref(_ffi.ArmScanDims(b, d, L, n, 1)), u.data_ptr(), dl.data_ptr(),
            A.data_ptr(), B.data_ptr(), B.data_ptr(), None, None, None, 1, 0, 0, 0,
            out.data_ptr(), None, None, torch.cuda.current_stream().cuda_stream)
    assert rc == 6 and _node_types(g.raw_cuda_graph()) == set()
