"""What a user of this framework has it do, as cases that can be timed and checked.

A case is a dict of plain values. `kind` says which path it takes, the rest are its sizes
and options. Sizes are those of the repository's configurations, tests and benchmark, or
generic ones of the same ranges. All tensors are float32 on the GPU, the one data type the
kernels compute in.

  step     one decode token of a Mamba-1 mixer: the convolution's step and the scan's
  seam     the convolution and the scan of one Mamba-1 layer at prefill, called as the
           Hugging Face mixer does: views of the projections in, time-major out
  scan     the Mamba-1 scan alone, contiguous rows, forward or reverse, with its options
  bidir    both time directions of one input, summed (vision and audio encoders)
  ss2d     the four-direction 2D cross-scan, one B and C per direction
  siso     the Mamba-3 SISO scan, from cos/sin or raw angles
  mimo     the Mamba-3 rank-r scan
  grid3    the Mamba-3 recurrence over a token grid: four causal traversals, or every
           position over every other one
  mixer    a whole Mamba-3 mixer: projection, gates, scan, projection
"""

import math

import torch
import torch.nn.functional as F

import armhackathon_amd as arm_scan

F32, F64 = torch.float32, torch.float64


def listed():
    return [
        # greedy generation at batch 1: one layer's two recurrent steps for one token
        dict(name="step_b1", kind="step", batch=1, dim=1536, state=16),
        # the same for a batch of requests that a server decodes together
        dict(name="step_b128", kind="step", batch=128, dim=1536, state=16),
        # a short chat prompt, of a length that is no multiple of anything
        dict(name="seam_b1_l77", kind="seam", batch=1, dim=1536, length=77, state=16),
        # a few requests of ordinary, odd length
        dict(name="seam_b4_l1531", kind="seam", batch=4, dim=1536, length=1531, state=16),
        # the benchmark's layer: Mamba-130M prefill, batch 8 x 2048 tokens
        dict(name="seam_b8_l2048", kind="seam", batch=8, dim=1536, length=2048, state=16),
        # one long document, streamed: few rows, many steps
        dict(name="scan_b1_l131072", kind="scan", batch=1, dim=768, length=131072, state=16,
             groups=1, reverse=False, softplus=True, z=True, resume=True),
        # an image as a sequence of 196 patches and a class token, both directions
        dict(name="bidir_b16_l197", kind="bidir", batch=16, dim=192, length=197, state=16),
        # a feature map of 64 x 64 tokens, four directions
        dict(name="ss2d_b16_64x64", kind="ss2d", batch=16, dim=192, height=64, width=64,
             state=16),
        # Mamba-3 prefill at batch 4, heads with queries and keys of their own
        dict(name="siso_b4_l4096", kind="siso", batch=4, length=4096, heads=24, dv=64, dqk=128,
             groups=24, angles=False, reverse=False, z=False, carry=True),
        # the same sizes at rank 4
        dict(name="mimo_b4_l4096", kind="mimo", batch=4, length=4096, heads=24, dv=64, dqk=128,
             groups=24, rank=4, angles=False, reverse=False, z=False, carry=True),
        # a small batch of token grids on the Mamba-3 recurrence, as a vision block has them
        dict(name="grid3_b2_28x28", kind="grid3", batch=2, height=28, width=28, heads=6, dv=32,
             dqk=64, causal=True),
        # a whole mixer of the published dimensions on one prompt
        dict(name="mixer_b1_l1024", kind="mixer", batch=1, length=1024, d_model=768,
             d_state=128, headdim=64, rank=1),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["step", "seam", "seam", "scan", "scan", "bidir", "ss2d", "siso", "siso",
                       "mimo", "grid3", "mixer"])
    flag = lambda: rng.random() < 0.5  # noqa: E731
    if kind == "step":
        return dict(kind=kind, batch=_log(rng, 1, 256), dim=rng.choice([768, 1536, 2048]),
                    state=16)
    if kind == "seam":
        batch = _log(rng, 1, 8)
        return dict(kind=kind, batch=batch, dim=1536, length=_log(rng, 16, 16384 // batch),
                    state=16)
    if kind == "scan":
        batch = _log(rng, 1, 16)
        dim = rng.choice([192, 384, 768, 1536])
        return dict(kind=kind, batch=batch, dim=dim,
                    length=_log(rng, 32, min(65536, 25000000 // (batch * dim))),
                    state=rng.choice([8, 16, 16]), groups=rng.choice([1, 1, 2]),
                    reverse=flag(), softplus=flag(), z=flag(), resume=flag())
    if kind == "bidir":
        batch = _log(rng, 1, 32)
        return dict(kind=kind, batch=batch, dim=rng.choice([192, 384, 768]),
                    length=_log(rng, 49, 4096 if batch <= 8 else 1024), state=16)
    if kind == "ss2d":
        side = _log(rng, 7, 64)
        other = max(7, min(64, side + rng.choice([0, 0, 0, -5, 3])))
        return dict(kind=kind, batch=_log(rng, 1, 16),
                    dim=192 if side > 28 else rng.choice([192, 384, 768]), height=side,
                    width=other, state=16)
    if kind in ("siso", "mimo"):
        batch = _log(rng, 1, 4)
        heads = rng.choice([8, 12, 24])
        case = dict(kind=kind, batch=batch, length=_log(rng, 64, 8192 // batch), heads=heads,
                    dv=64, dqk=rng.choice([64, 128, 128]), groups=rng.choice([1, 1, heads]))
        if kind == "mimo":
            case.update(rank=rng.choice([2, 4, 4]))
        reverse = rng.random() < 0.25
        case.update(angles=flag(), reverse=reverse, z=flag(), carry=flag())
        return case
    if kind == "grid3":
        return dict(kind=kind, batch=_log(rng, 1, 4), height=_log(rng, 7, 48),
                    width=_log(rng, 7, 48), heads=rng.choice([3, 6]), dv=32, dqk=64,
                    causal=flag())
    batch = _log(rng, 1, 4)
    return dict(kind=kind, batch=batch, length=_log(rng, 64, 8192 // batch), d_model=768,
                d_state=128, headdim=64, rank=rng.choice([1, 1, 4]))


# ----------------------------------------------------------------------- inputs
class _Draw:
    """Seeded draws on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, *shape, mean=0.0, std=1.0):
        x = torch.randn(shape, generator=self.g, device="cuda")
        return x if std == 1.0 and mean == 0.0 else x.mul_(std).add_(mean)

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, generator=self.g, device="cuda").mul_(hi - lo).add_(lo)


def _m1_weights(r, dim, state):
    """A as Mamba initialises it, -1 .. -state for every channel; D and the bias of dt."""
    a = -torch.arange(1, state + 1, dtype=F32, device="cuda").repeat(dim, 1)
    return a, r.normal(dim), r.uniform(-0.5, 0.5, dim)


def _mixer_module(case, seed):
    from armhackathon_amd.mamba3_block import Mamba3Mixer

    r = _Draw(seed)
    m = Mamba3Mixer(d_model=case["d_model"], d_state=case["d_state"], headdim=case["headdim"],
                    is_mimo=case["rank"] > 1, mimo_rank=case["rank"]).to("cuda")
    with torch.no_grad():
        for name, p in m.named_parameters():
            if name.endswith("proj.weight"):
                p.copy_(r.normal(*p.shape, std=p.shape[1] ** -0.5))
            elif name == "dt_bias":
                p.copy_(r.uniform(-4.0, -2.0, *p.shape))
            else:  # the norms, D, the biases of B and C and the rank maps
                p.mul_(1.0 + 0.2 * r.normal(*p.shape))
    return m.requires_grad_(False)


def _m3_inputs(case, seed):
    """The Mamba-3 scan's inputs: dt = softplus(N(0,1) - 4), A < 0 per head, rotation
    angles that grow with dt, queries and keys of unit length."""
    r = _Draw(seed)
    b, length, h, dv, dqk, g = (case[k] for k in ("batch", "length", "heads", "dv", "dqk",
                                                  "groups"))
    rank = (case["rank"],) if case["kind"] == "mimo" else ()
    dt = F.softplus(r.normal(b, h, length, mean=-4.0))
    t = dict(dt=dt, trap=r.normal(b, h, length))
    t["adt"] = -torch.exp(r.normal(h, std=0.5))[None, :, None] * dt
    t["q"] = r.normal(b, length, *rank, g, dqk, std=dqk ** -0.5)
    t["k"] = r.normal(b, length, *rank, g, dqk, std=dqk ** -0.5)
    t["v"] = r.normal(b, length, h, dv)
    t["q_bias"] = r.normal(h, *rank, dqk, std=0.1)
    t["k_bias"] = r.normal(h, *rank, dqk, std=0.1)
    if case["angles"]:
        t["angles"] = r.normal(b, length, h, dqk // 4)
    else:
        theta = r.uniform(-math.pi, math.pi, b, length, h, dqk // 2)
        theta = theta.mul_(dt.transpose(1, 2)[..., None]).double().cumsum_(1)
        t["cos"], t["sin"] = theta.cos().float(), theta.sin().float()
    t["D"] = r.normal(h)
    if case["z"]:
        t["z"] = r.normal(b, length, h, dv)
    if rank:
        for name in ("psi", "zeta", "phi"):
            t[name] = r.normal(h, *rank, dv, std=0.5)
    return t


def prepare(case, seed):
    kind = case["kind"]
    r = _Draw(seed)
    if kind == "step":
        b, d, n = case["batch"], case["dim"], case["state"]
        a, skip, bias = _m1_weights(r, d, n)
        # the mixer's views: x and z are halves of one projection, B and C columns of another
        xz, dbc = r.normal(b, 2 * d), r.normal(b, 48 + 2 * n)
        t = dict(x=xz[:, :d], z=xz[:, d:], dt=r.normal(b, d, mean=-4.0, std=0.5), A=a, D=skip,
                 bias=bias, B=dbc[:, 48:48 + n], C=dbc[:, 48 + n:],
                 conv_state=r.normal(b, d, 4), conv_weight=r.normal(d, 4, std=0.5),
                 conv_bias=r.normal(d, std=0.1), state=r.normal(b, d, n, std=0.1))
    elif kind == "seam":
        b, d, length, n = case["batch"], case["dim"], case["length"], case["state"]
        a, skip, bias = _m1_weights(r, d, n)
        x, z = r.normal(b, length, 2 * d).transpose(1, 2).chunk(2, dim=1)
        dbc = r.normal(b, length, 48 + 2 * n)
        t = dict(x=x, z=z, delta=r.normal(b, d, length, mean=-4.0, std=0.5), A=a, D=skip,
                 bias=bias, B=dbc[..., 48:48 + n].transpose(1, 2),
                 C=dbc[..., 48 + n:].transpose(1, 2), conv_weight=r.normal(d, 4, std=0.5),
                 conv_bias=r.normal(d, std=0.1))
    elif kind in ("scan", "bidir"):
        b, d, length, n = case["batch"], case["dim"], case["length"], case["state"]
        g = case.get("groups", 1)
        a, skip, bias = _m1_weights(r, d, n)
        t = dict(u=r.normal(b, d, length), delta=r.normal(b, d, length, mean=-4.0, std=0.5),
                 A=a, B=r.normal(b, g, n, length), C=r.normal(b, g, n, length), D=skip)
        if case.get("softplus", True):
            t["bias"] = bias
        else:
            t["delta"] = F.softplus(t["delta"])
        if case.get("z", True):
            t["z"] = r.normal(b, d, length)
        if case.get("resume"):
            t["h0"] = r.normal(b, d, n, std=0.1)
    elif kind == "ss2d":
        b, d, n, hh, ww = (case[k] for k in ("batch", "dim", "state", "height", "width"))
        a, skip, bias = _m1_weights(r, d, n)
        t = dict(u=r.normal(b, d, hh, ww), delta=r.normal(b, d, hh, ww, mean=-4.0, std=0.5),
                 A=a, B=r.normal(4, b, n, hh, ww), C=r.normal(4, b, n, hh, ww), D=skip,
                 bias=bias, z=r.normal(b, d, hh, ww))
    elif kind in ("siso", "mimo"):
        t = _m3_inputs(case, seed)
    elif kind == "grid3":
        b, hh, ww, h, dv, dqk = (case[k] for k in ("batch", "height", "width", "heads", "dv",
                                                   "dqk"))
        dt = F.softplus(r.normal(b, h, hh, ww, mean=-3.0, std=0.5))
        t = dict(q=r.normal(b, hh, ww, 1, dqk, std=dqk ** -0.5),
                 k=r.normal(b, hh, ww, 1, dqk, std=dqk ** -0.5), v=r.normal(b, hh, ww, h, dv),
                 dt=dt, trap=r.normal(b, h, hh, ww),
                 adt=-torch.exp(r.normal(h, std=0.5))[None, :, None, None] * dt,
                 angles=r.normal(b, hh, ww, h, dqk // 4), q_bias=r.normal(h, dqk, std=0.1),
                 k_bias=r.normal(h, dqk, std=0.1), D=r.normal(h), z=r.normal(b, hh, ww, h, dv))
    else:
        t = dict(module=_mixer_module(case, seed),
                 u=r.normal(case["batch"], case["length"], case["d_model"]))
    return case, t


# ----------------------------------------------------------------------- the paths
def run(state):
    case, t = state
    kind = case["kind"]
    if kind == "step":
        x = arm_scan.causal_conv1d_update(t["x"], t["conv_state"], t["conv_weight"],
                                          bias=t["conv_bias"], activation="silu")
        y = arm_scan.selective_state_update(t["state"], x, t["dt"], t["A"], t["B"], t["C"],
                                            D=t["D"], z=t["z"], dt_bias=t["bias"],
                                            dt_softplus=True)
        return y, t["conv_state"], t["state"]
    if kind == "seam":
        u = arm_scan.causal_conv1d(t["x"], t["conv_weight"], bias=t["conv_bias"],
                                   activation="silu", time_major=True)
        return arm_scan.selective_scan_time_major(
            u, t["delta"], t["A"], t["B"], t["C"], D=t["D"], z=t["z"], delta_bias=t["bias"],
            delta_softplus=True, return_last_state=True)
    if kind == "scan":
        return arm_scan.selective_scan(
            t["u"], t["delta"], t["A"], t["B"], t["C"], D=t["D"], z=t.get("z"),
            delta_bias=t.get("bias"), delta_softplus=case["softplus"], return_last_state=True,
            initial_state=t.get("h0"), reverse=case["reverse"])
    if kind == "bidir":
        return arm_scan.bidirectional_scan(
            t["u"], t["delta"], t["A"], t["B"], t["C"], D=t["D"], z=t["z"],
            delta_bias=t["bias"], delta_softplus=True, merge="sum")
    if kind == "ss2d":
        return arm_scan.ss2d_scan(t["u"], t["delta"], t["A"], t["B"], t["C"], D=t["D"],
                                  delta_bias=t["bias"], delta_softplus=True, z=t["z"],
                                  per_direction=True)
    if kind in ("siso", "mimo"):
        ranks = [t[k] for k in ("psi", "zeta", "phi")] if kind == "mimo" else []
        fn = arm_scan.mamba3_mimo_scan if ranks else arm_scan.mamba3_scan
        return fn(*[t[k] for k in ("q", "k", "v", "adt", "dt", "trap", "q_bias", "k_bias")],
                  *ranks, angles=t.get("angles"), cos=t.get("cos"), sin=t.get("sin"), D=t["D"],
                  z=t.get("z"), reverse=case["reverse"], return_last_state=case["carry"])
    if kind == "grid3":
        fn = arm_scan.ss2d_scan_mamba3 if case["causal"] else arm_scan.ss2d_noncausal_mamba3
        return fn(*[t[k] for k in ("q", "k", "v", "adt", "dt", "trap", "q_bias", "k_bias",
                                   "angles")], D=t["D"], z=t["z"])
    return t["module"](t["u"])


# ----------------------------------------------------------------------- their least work
def work(case):
    kind, b = case["kind"], case["batch"]
    if kind in ("step", "seam", "scan", "bidir", "ss2d"):
        d, n = case["dim"], case["state"]
        length = 1 if kind == "step" else (case["height"] * case["width"] if kind == "ss2d"
                                           else case["length"])
        row, g = b * d * length, case.get("groups", 1)
        # u (or x), delta, z and the output; B and C; A, D and the bias; the final states
        floats = row * (3 + int(case.get("z", True))) + d * (n + 2)
        floats += 2 * b * g * n * length * (4 if kind == "ss2d" else 1)
        if kind == "step":
            floats += 2 * b * d * (n + 4) + 5 * d  # both states read and written, the taps
        elif kind in ("seam", "scan"):
            floats += b * d * n * (2 if case.get("resume") else 1) + 5 * d * (kind == "seam")
        # per state: the decay's argument, the input, the update and the output (an
        # exponential besides); per step and channel the gate, the skip and the taps
        passes = {"bidir": 2, "ss2d": 4}.get(kind, 1)
        flops = passes * row * (7 * n + 8) + (8 * row if kind in ("step", "seam") else 0)
        return {"bytes": 4 * floats, "flops": flops}
    if kind == "mixer":
        heads = 2 * case["d_model"] // case["headdim"]
        inner, n, rank = 2 * case["d_model"], case["d_state"], case["rank"]
        width = 2 * inner + 2 * n * rank + 3 * heads + n // 4
        tokens = b * case["length"]
        weights = case["d_model"] * (width + inner) + 2 * heads * rank * n
        flops = 2 * tokens * case["d_model"] * (width + inner) + 4 * tokens * rank * inner * n
        return {"bytes": 4 * (2 * tokens * case["d_model"] + weights), "flops": flops}
    h, dv, dqk = case["heads"], case["dv"], case["dqk"]
    rank, length = case.get("rank", 1), case.get("length", 0)
    if kind == "grid3":
        length, passes, group = case["height"] * case["width"], 4, 1
        rot, gate, carry = dqk // 4, 1, 0
    else:
        passes, group, gate, carry = 1, case["groups"], int(case["z"]), int(case["carry"])
        rot = dqk // 4 if case["angles"] else dqk  # raw angles, or cos and sin
    floats = b * length * (2 * rank * group * dqk + h * (rot + dv * (2 + gate) + 3))
    floats += carry * b * h * dv * dqk + 2 * h * rank * dqk + 3 * h * rank * dv * (rank > 1)
    # the state's update and its read-out, a multiply and an add each
    return {"bytes": 4 * floats, "flops": passes * 4 * b * length * h * rank * dv * dqk}


def tolerance(case):
    # Everything is summed in 32 bits. Measured against 64-bit sums (2-norm, and the largest
    # difference over the root mean square): the Mamba-1 paths 0.6e-7 to 1.9e-7 and up to
    # 3e-6, Mamba-3 0.3e-7 to 4.4e-7 and up to 1e-5 (the states at rank 4 the largest), the
    # mixer, whose projections are 32-bit products of 768 and 1536 terms, 1.2e-6 and 9e-6.
    # About four times that.
    if case["kind"] == "mixer":
        return {"rel": 5e-6, "max": 4e-5}
    if case["kind"] in ("siso", "mimo", "grid3"):
        return {"rel": 2e-6, "max": 4e-5}
    return {"rel": 8e-7, "max": 1.2e-5}


# ----------------------------------------------------------------------- 64-bit results
def _scan64(u, delta, A, B, C, D=None, z=None, bias=None, softplus=True, reverse=False,
            h0=None):
    """The Mamba-1 recurrence step by step: u, delta, z (b, d, L), B, C (b, g, n, L)."""
    u, delta, A, B, C = u.to(F64), delta.to(F64), A.to(F64), B.to(F64), C.to(F64)
    b, d, length = u.shape
    g = B.shape[1]
    if bias is not None:
        delta = delta + bias.to(F64)[:, None]
    if softplus:
        delta = F.softplus(delta)
    h = torch.zeros(b, d, A.shape[1], dtype=F64, device=u.device) if h0 is None else h0.to(F64)
    y = torch.empty_like(u)
    block = max(1, min(length, (1 << 28) // h.numel()))
    starts = list(range(0, length, block))
    for s in (reversed(starts) if reverse else starts):
        e = min(length, s + block)
        dt = delta[:, :, s:e].permute(2, 0, 1).unsqueeze(-1)  # (T, b, d, 1)
        decay = torch.exp(dt * A)
        per_channel = lambda m: m[..., s:e].permute(3, 0, 1, 2).repeat_interleave(  # noqa: E731
            d // g, dim=2)
        hs = dt * u[:, :, s:e].permute(2, 0, 1).unsqueeze(-1) * per_channel(B)
        steps = range(e - s - 1, -1, -1) if reverse else range(e - s)
        for t in steps:
            h = torch.addcmul(hs[t], decay[t], h, out=hs[t])
        h = h.clone()
        y[:, :, s:e] = (hs * per_channel(C)).sum(-1).permute(1, 2, 0)
        del decay, hs
    if D is not None:
        y = y + u * D.to(F64)[:, None]
    if z is not None:
        y = y * F.silu(z.to(F64))
    return y, h


def _rotate64(x, cos, sin, split):
    """Pairs (i, i + half) when split, else (2i, 2i + 1)."""
    if split:
        a, c = x.chunk(2, dim=-1)
        return torch.cat((a * cos - c * sin, a * sin + c * cos), dim=-1)
    a, c = x[..., 0::2], x[..., 1::2]
    return torch.stack((a * cos - c * sin, a * sin + c * cos), dim=-1).flatten(-2)


def _angles64(angles, dt, half):
    theta = torch.cumsum(torch.tanh(angles.to(F64)) * math.pi
                         * dt.to(F64).transpose(1, 2)[..., None], dim=1)
    theta = F.pad(theta, (0, half - theta.shape[-1]))
    return theta.cos(), theta.sin()


def _m3_64(t, reverse=False, same_step=True):
    """The Mamba-3 recurrence step by step -> out (b, L, h, dv), state (b, h, dv, dqk), the
    last step's input. Without same_step, a step's own key and D stay out of its output."""
    mimo = "psi" in t
    v, dt = t["v"].to(F64), t["dt"].to(F64)
    b, length, h, dv = v.shape
    q, k = t["q"].to(F64), t["k"].to(F64)
    if not mimo:
        q, k = q.unsqueeze(2), k.unsqueeze(2)
    rank, g, dqk = q.shape[2:]
    if t.get("cos") is None:
        cos, sin = _angles64(t["angles"], dt, dqk // 2)
    else:
        cos, sin = t["cos"].to(F64), t["sin"].to(F64)
    per_head = lambda x, bias: _rotate64(  # noqa: E731
        x.repeat_interleave(h // g, dim=3) + bias.to(F64).reshape(h, rank, dqk).transpose(0, 1),
        cos.unsqueeze(2), sin.unsqueeze(2), mimo)
    q, k = per_head(q, t["q_bias"]), per_head(k, t["k_bias"])  # (b, L, r, h, dqk)
    if mimo:
        psi, zeta, phi = (t[n].to(F64).transpose(0, 1) for n in ("psi", "zeta", "phi"))
        x = v.unsqueeze(2) * psi
    else:
        x = v.unsqueeze(2)
    lam = torch.sigmoid(t["trap"].to(F64))
    gamma, carry = dt * lam, dt * (1.0 - lam)
    scale = gamma.clone()  # a step's input also carries its neighbour's share
    if reverse:
        scale[..., 1:] += carry[..., :-1]
    else:
        scale[..., :-1] += carry[..., 1:]
    alpha = torch.exp(t["adt"].to(F64))
    # per step: (b h, r, .) matrices
    rows = lambda m: m.permute(1, 0, 3, 2, 4).reshape(length, b * h, rank, -1)  # noqa: E731
    qs, ks, xs = rows(q), rows(k), rows(x)
    kt = ks.transpose(2, 3).contiguous()
    per = lambda m: m.permute(2, 0, 1).reshape(length, b * h, 1, 1)  # noqa: E731
    al, ga, sc = per(alpha), per(gamma), per(scale)
    xsc = sc * xs
    s = torch.zeros(b * h, dqk, dv, dtype=F64, device=v.device)
    read = torch.empty(length, b * h, rank, dv, dtype=F64, device=v.device)
    for i in (range(length - 1, -1, -1) if reverse else range(length)):
        s.mul_(al[i])
        torch.matmul(qs[i], s, out=read[i])
        s.baddbmm_(kt[i], xsc[i])
    if same_step:
        read += ga * torch.matmul(torch.matmul(qs, kt), xs)
        if t.get("D") is not None:
            read += t["D"].to(F64).repeat(b)[:, None, None] * xs
    y = read.reshape(length, b, h, rank, dv).permute(1, 0, 3, 2, 4)  # (b, L, r, h, dv)
    z = None if t.get("z") is None else t["z"].to(F64).unsqueeze(2)
    if mimo:
        y = y * phi
    if z is not None:
        y = y * F.silu(z * zeta if mimo else z)
    end = 0 if reverse else length - 1
    last = (sc[end] * ks[end]).reshape(b, h, rank, dqk)[:, :, 0]
    return y.sum(2), s.transpose(1, 2).reshape(b, h, dv, dqk), last


def _grid64(t, causal):
    b, hh, ww = t["q"].shape[:3]
    total = 0
    for columns in (False, True):
        tm = lambda x: (x.transpose(1, 2) if columns else x).reshape(  # noqa: E731
            b, hh * ww, *x.shape[3:])
        hm = lambda x: (x.transpose(2, 3) if columns else x).reshape(b, -1, hh * ww)  # noqa: E731
        o = {n: tm(t[n]) for n in ("q", "k", "v", "angles", "z")}
        o.update({n: hm(t[n]) for n in ("adt", "dt", "trap")})
        o.update({n: t[n] for n in ("q_bias", "k_bias", "D")})
        y = _m3_64(o)[0] + _m3_64(o, reverse=True, same_step=causal)[0]
        total = total + (y.reshape(b, ww, hh, *y.shape[2:]).transpose(1, 2) if columns
                         else y.reshape(b, hh, ww, *y.shape[2:]))
    return total


def _mixer64(case, m, u):
    u = u.to(F64)
    b, length, _ = u.shape
    heads, rank, n = m.nheads, case["rank"], case["d_state"]
    z, x, B, C, ddt, dda, trap, ang = torch.split(u @ m.in_proj.weight.to(F64).T,
                                                  m.split_sizes, dim=-1)
    norm = lambda v, w: (v := v.reshape(b, length, rank, 1, n)) * torch.rsqrt(  # noqa: E731
        v.square().mean(-1, keepdim=True) + 1e-5) * w.to(F64)
    dt = F.softplus(ddt + m.dt_bias.to(F64))
    decay = torch.where(dda >= 0, 1.0 + dda, 1.0 / (1.0 - dda.clamp_max(0.0)))
    adt = torch.clamp_max(-decay, -m.A_floor) * dt
    t = dict(q=norm(C, m.C_norm.weight), k=norm(B, m.B_norm.weight),
             v=x.reshape(b, length, heads, -1), z=z.reshape(b, length, heads, -1),
             adt=adt.transpose(1, 2), dt=dt.transpose(1, 2), trap=trap.transpose(1, 2),
             angles=ang.unsqueeze(2).expand(b, length, heads, ang.shape[-1]),
             q_bias=m.C_bias, k_bias=m.B_bias, D=m.D)
    if rank > 1:
        t.update(psi=m.mimo_x, zeta=m.mimo_z, phi=m.mimo_o)
    else:
        t["q"], t["k"] = t["q"][:, :, 0], t["k"][:, :, 0]
    y = _m3_64(t)[0].reshape(b, length, -1)
    return y @ m.out_proj.weight.to(F64).T


def exact(case, seed):
    _, t = prepare(case, seed)
    kind = case["kind"]
    if kind == "step":
        window = torch.cat((t["conv_state"][..., 1:], t["x"].unsqueeze(-1)), dim=-1)
        x = F.silu((window.to(F64) * t["conv_weight"].to(F64)).sum(-1) + t["conv_bias"].to(F64))
        y, h = _scan64(x.unsqueeze(-1), t["dt"].unsqueeze(-1), t["A"],
                       t["B"][:, None, :, None], t["C"][:, None, :, None], t["D"],
                       t["z"].unsqueeze(-1), t["bias"], h0=t["state"])
        return y.squeeze(-1), window, h
    if kind == "seam":
        x = F.pad(t["x"].to(F64), (3, 0))
        length, w = case["length"], t["conv_weight"].to(F64)
        u = sum(w[:, i, None] * x[..., i:i + length] for i in range(4))
        u = F.silu(u + t["conv_bias"].to(F64)[:, None])
        return _scan64(u, t["delta"], t["A"], t["B"].unsqueeze(1), t["C"].unsqueeze(1), t["D"],
                       t["z"], t["bias"])
    if kind == "scan":
        return _scan64(t["u"], t["delta"], t["A"], t["B"], t["C"], t["D"], t.get("z"),
                       t.get("bias"), case["softplus"], case["reverse"], t.get("h0"))
    if kind == "bidir":
        return sum(_scan64(t["u"], t["delta"], t["A"], t["B"], t["C"], t["D"], t["z"],
                           t["bias"], True, rev)[0] for rev in (False, True))
    if kind == "ss2d":
        total = 0
        for i, rev in enumerate((False, True, False, True)):
            seq = lambda x, c=i >= 2: (x.transpose(-1, -2) if c else x).flatten(-2)  # noqa: E731
            y, _ = _scan64(seq(t["u"]), seq(t["delta"]), t["A"], seq(t["B"][i]).unsqueeze(1),
                           seq(t["C"][i]).unsqueeze(1), t["D"], seq(t["z"]), t["bias"], True,
                           rev)
            b, d, hh, ww = t["u"].shape
            total = total + (y.reshape(b, d, ww, hh).transpose(2, 3) if i >= 2
                             else y.reshape(b, d, hh, ww))
        return total
    if kind in ("siso", "mimo"):
        out, state, last = _m3_64(t, reverse=case["reverse"])
        if not case["carry"]:
            return out
        return (out, state, last) if kind == "siso" else (out, state)
    if kind == "grid3":
        return _grid64(t, case["causal"])
    return _mixer64(case, t["module"], t["u"])
