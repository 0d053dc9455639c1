"""The work that users of dnsjax_amd have it do, as measured cases.

Every case is one call, or one short sequence of calls, through the public
entry points, on inputs a program would have at hand: a seeded solenoidal
velocity field, the flow object (native context) that the program keeps
through its run, and, where it trains or uses a network, that network.
``exact`` restates each case in plain torch, in 64 bits.

Kinds:
  step      one time step by the ``make_stepper`` pair as a drop-in caller
            writes it: predict_and_correct, one iterate_correction,
            correct_velocity
  run       the driver's time loop (corrector to tolerance, the error read on
            the host) with its energy record
  guess     a step started from the corrector guess (extrapolation, or the
            per-mode network), two corrector passes, correct_velocity
  ensemble  one device-decided step of several trajectories in one batch plan
  pgrad     gradient of the profile network for one training batch
  pforward  the profile network's output for every Fourier mode of a flow
  mgrad     gradient of the per-mode network for one training batch
"""

from __future__ import annotations

import math

import torch

from dnsjax_amd import learned, profile_net
from dnsjax_amd.driver import StatsRecorder
from dnsjax_amd.driver import run as run_driver
from dnsjax_amd.flows import make_flow
from dnsjax_amd.native import BatchPlan
from dnsjax_amd.params import Params

F64, C128 = torch.float64, torch.complex128
DEV = "cuda"


def _periodic(kind, n, **kw):
    nx, ny, nz = n if isinstance(n, tuple) else (n, n, n)
    c = dict(kind=kind, system="kolmogorov", nx=nx, ny=ny, nz=nz, re=100.0, dt=0.005, rms=0.1, tilt=0.0,
             implicitness=0.5, oversample_y=True, precision="fp64")
    c.update(kw)
    return c


def _couette(kind, nx, ny, nz, **kw):
    c = dict(kind=kind, system="plane-couette", nx=nx, ny=ny, nz=nz, re=400.0, dt=0.01, rms=0.05, p=4,
             implicitness=0.5, precision="fp64")
    c.update(kw)
    return c


def listed():
    return [
        # the smallest flow anyone runs: launches and latency count
        dict(_periodic("step", 32, re=40.0, dt=0.01, rms=0.01), name="kolmogorov 32 fp64 step"),
        # the benchmark flow in the plain method, the largest cube supported
        dict(_periodic("step", 128), name="kolmogorov 128 fp64 step"),
        # the benchmark flow in its fastest form: mixed precision, cubic guess
        dict(_periodic("guess", 128, precision="mixed", mode=4), name="kolmogorov 128 mixed guess"),
        # uneven box, tilted forcing, no oversampling in y, off-centre scheme
        dict(_periodic("step", (96, 64, 48), system="waleffe", tilt=30.0, oversample_y=False, implicitness=0.6,
                       precision="mixed"), name="waleffe 96x64x48 mixed step"),
        # a small production run as the driver does it, energies recorded
        dict(_periodic("run", 64, steps=2), name="kolmogorov 64 fp64 run"),
        # an ensemble's size class: 16 trajectories per launch
        dict(_periodic("ensemble", 48, re=40.0, dt=0.01, rms=0.05, precision="mixed", members=16, slots=5),
             name="ensemble 16x48 mixed"),
        # plane Couette at its usual size
        dict(_couette("step", 64, 128, 64), name="couette 64x128x64 fp64 step"),
        # plane Couette at its largest, sixth-order differences
        dict(_couette("step", 128, 256, 128, re=1000.0, dt=0.005, p=6), name="couette 128x256x128 fp64 step"),
        # a small channel with odd ny, mixed, started from the learned guess
        dict(_couette("guess", 48, 65, 32, precision="mixed", mode=2, hidden=32), name="couette 48x65x32 mixed guess"),
        # training the wall-normal profile network: one mini-batch
        dict(kind="pgrad", ny=256, hidden=256, batch=2048, name="profile net gradient"),
        # the same network over all modes of the 128x256x128 flow
        dict(kind="pforward", ny=256, hidden=256, batch=8128, name="profile net forward"),
        # training the per-mode network: one mini-batch
        dict(kind="mgrad", hidden=32, batch=8192, bf16=True, name="mode net gradient"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "guess", "run", "ensemble", "couette", "couette", "cguess", "pgrad", "pforward",
                       "mgrad"])
    sizes = (16, 32, 48, 64, 96, 128)
    if kind in ("step", "guess", "run", "ensemble"):
        flow = dict(system=rng.choice(["kolmogorov", "kolmogorov", "waleffe"]), re=round(rng.uniform(20.0, 150.0), 2),
                    dt=round(rng.uniform(0.002, 0.01), 4), rms=round(rng.uniform(0.01, 0.1), 3),
                    precision=rng.choice(["fp64", "mixed"]))
        if kind == "ensemble":
            n = tuple(rng.choice((16, 32, 48, 64)) for _ in range(3))
            return _periodic(kind, n, members=rng.randint(2, 16), slots=5, **flow)
        n = tuple(rng.choice(sizes) for _ in range(3))
        if kind == "step":
            flow["tilt"] = rng.choice([0.0, 0.0, round(rng.uniform(1.0, 89.0), 1)])
            flow["oversample_y"] = n[1] in (48, 96) or rng.random() < 0.7
            flow["implicitness"] = rng.choice([0.5, 0.5, round(rng.uniform(0.4, 1.0), 2)])
        elif kind == "guess":
            flow["mode"] = rng.choice([1, 3, 4])
        else:
            flow["steps"] = rng.randint(1, 3)
        return _periodic(kind, n, **flow)
    if kind in ("couette", "cguess"):
        nx, nz = rng.choice(sizes), rng.choice(sizes)
        flow = dict(re=round(rng.uniform(200.0, 1000.0), 1), dt=round(rng.uniform(0.004, 0.01), 4),
                    p=rng.choice([2, 4, 6, 8]), precision=rng.choice(["fp64", "mixed"]))
        ny = _log_int(rng, 24, 256)
        if kind == "couette":
            return _couette("step", nx, ny, nz, **flow)
        return _couette("guess", nx, ny, nz, mode=rng.choice([2, 3]), hidden=rng.choice([32, 64]), **flow)
    if kind == "mgrad":
        return dict(kind=kind, hidden=rng.choice([32, 64]), batch=_log_int(rng, 256, 16384), bf16=rng.random() < 0.8)
    return dict(kind=kind, ny=_log_int(rng, 32, 256), hidden=rng.choice([64, 128, 256]),
                batch=_log_int(rng, 256, 2048 if kind == "pgrad" else 8128))


# ---------------------------------------------------------------- inputs
def _params(c, **kw):
    common = dict(system=c["system"], nx=c["nx"], ny=c["ny"], nz=c["nz"], re=c["re"], dt=c["dt"],
                  implicitness=c["implicitness"], precision=c["precision"])
    if c["system"] == "plane-couette":
        common.update(lx=2 * math.pi, lz=math.pi, fd_order=c["p"], corrector_tolerance=1e-8)
    else:
        common.update(lx=2 * math.pi, ly=2 * math.pi, lz=2 * math.pi, tilt_degree=c["tilt"],
                      oversample_y=c["oversample_y"], corrector_tolerance=1e-10)
    common.update(kw)
    return Params(**common)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _harmonics(n, stored):
    """Stored full-axis harmonics 0 .. n/2-1, -(n/2-1) .. -1."""
    i = torch.arange(stored, device=DEV, dtype=F64)
    return torch.where(i < n // 2, i, i - (n - 1))


def _negated(n1):
    """Index of the opposite harmonic on a stored full axis."""
    return (n1 - torch.arange(n1, device=DEV)) % n1


def _spectrum(k):
    return k**4 * torch.exp(-2.0 * (k / 4.0) ** 2)


def _field(c, seed):
    """A seeded velocity perturbation of the case's RMS: solenoidal with
    E(k) ~ k^4 exp(-2 (k/4)^2) (periodic), or the curl of such a potential
    under a (1 - y^2)^2 envelope, no-slip (plane Couette)."""
    g = _gen(seed)
    hx = torch.arange(c["nx"] // 2, device=DEV, dtype=F64)
    hz = _harmonics(c["nz"], c["nz"] - 1)
    if c["system"] != "plane-couette":
        hy = _harmonics(c["ny"], c["ny"] - 1)
        k = torch.stack(torch.broadcast_tensors(hx.view(1, 1, -1), hy.view(-1, 1, 1), hz.view(1, -1, 1)))
        k2 = (k * k).sum(0)
        safe = torch.where(k2 > 0, k2, 1.0)
        amp = torch.where(k2 > 0, torch.sqrt(_spectrum(safe.sqrt()) / (4 * math.pi * safe)), 0.0)
        u = torch.randn((3,) + k2.shape, generator=g, device=DEV, dtype=C128) * amp
        u = u - k * ((k * u).sum(0) / safe)
        iy, iz = _negated(c["ny"] - 1), _negated(c["nz"] - 1)
        u[..., 0] = (u[..., 0] + u[..., 0][:, iy][:, :, iz].conj()) / 2
        u[:, 0, 0, 0] = 0
        km = torch.where(hx == 0, 1.0, 2.0)
        ep = 0.5 * (km * (u.abs() ** 2)).sum()
    else:
        ny = c["ny"]
        y = _cgl(ny)
        k = torch.sqrt(hx.view(1, -1) ** 2 + hz.view(-1, 1) ** 2)
        safe = torch.where(k > 0, k, 1.0)
        amp = torch.where(k > 0, torch.sqrt(_spectrum(safe) / (2 * math.pi * safe)), 0.0)
        m = torch.arange(8, device=DEV, dtype=F64)
        a = torch.randn((3,) + k.shape + (8,), generator=g, device=DEV, dtype=C128)
        a = a * amp[..., None] * torch.exp(-m / 4)
        th = torch.acos(y.clamp(-1, 1))
        T = torch.cos(m[:, None] * th)
        sin = torch.sin(th).clamp_min(1e-300)
        dT = m[:, None] * torch.sin(m[:, None] * th) / sin
        dT[:, 0] = m * m * (-1.0) ** (m + 1)
        dT[:, -1] = m * m
        env, denv = (1 - y * y) ** 2, -4 * y * (1 - y * y)
        psi = (a @ T.to(C128)) * env
        dpsi = (a @ (T * denv + dT * env).to(C128))
        kx, kz = (2 * math.pi / (2 * math.pi)) * hx.view(1, -1, 1), (2 * math.pi / math.pi) * hz.view(-1, 1, 1)
        u = torch.stack([dpsi[2] - 1j * kz * psi[1], 1j * kz * psi[0] - 1j * kx * psi[2],
                         1j * kx * psi[1] - dpsi[0]])
        iz = _negated(c["nz"] - 1)
        u[:, :, 0] = (u[:, :, 0] + u[:, iz, 0].conj()) / 2
        u[..., 0] = u[..., -1] = 0
        km = torch.where(hx == 0, 1.0, 2.0).view(1, 1, -1, 1)
        ep = 0.5 * ((km * u.abs() ** 2).sum((0, 1, 2)) * _quadrature(y)).sum() / 2.0
    return (u * (c["rms"] / torch.sqrt(2 * ep / 3))).contiguous()


def _history(c, n0, seed):
    """Earlier nonlinear terms of a smooth trajectory that ends at n0, newest
    first, as the (re, im) FP32 fields that the guess keeps."""
    g = _gen(seed)
    trend = 1e-3 * torch.randn(n0.shape[0], 1, 1, 1, generator=g, device=DEV, dtype=F64)
    noise = torch.randn(n0.shape, generator=g, device=DEV, dtype=C128)
    return [torch.view_as_real(n0 * (1 - j * trend - 1e-5 * j * j * noise.real)).float().contiguous()
            for j in (1, 2, 3)]


def _net_inputs(c, seed):
    g = _gen(seed)
    if c["kind"] == "mgrad":
        X = torch.randn(c["batch"], 16, generator=g, device=DEV)
        return X, torch.randn(c["batch"], 6, generator=g, device=DEV)
    X = torch.randn(c["batch"], profile_net.profile_din(c["ny"]), generator=g, device=DEV)
    X[:, 12 * c["ny"] + 3:] = 0
    T = torch.randn(c["batch"], 6 * c["ny"], generator=g, device=DEV) if c["kind"] == "pgrad" else None
    return X.to(torch.bfloat16), T


def _some_biases(net, seed):
    """Biases as training leaves them (they start at zero)."""
    g = _gen(seed + 7)
    for b in net.unpack()[1::2]:
        b.copy_(0.1 * torch.randn(b.shape, generator=g, device=DEV))


SCALES = (50.0, 500.0, 1e-3)  # feature scales 1/rms(D1), 1/rms(D2) and the residual's rms


def _member(c, i, seed):
    """Case of ensemble member i: its own Reynolds number and field."""
    return dict(c, re=c["re"] * (0.5 + i / c["members"]))


def _mode_net(c, seed):
    net = learned.Net(c["hidden"], seed=seed)
    _some_biases(net, seed)
    net.pack()
    return net


def prepare(case, seed):
    c = case
    kind = c["kind"]
    if kind in ("pgrad", "pforward"):
        net = profile_net.ProfileNet(c["ny"], c["hidden"], seed=seed)
        _some_biases(net, seed)
        X, T = _net_inputs(c, seed)
        return dict(kind=kind, net=net, X=X.view(torch.int16), T=T)
    if kind == "mgrad":
        net = learned.Net(c["hidden"], seed=seed)
        _some_biases(net, seed)
        X, T = _net_inputs(c, seed)
        return dict(kind=kind, net=net, X=X, T=T, bf16=c["bf16"])
    if kind == "ensemble":
        flows = []
        for i in range(c["members"]):
            # one size class: the members run the kernels its first one chose
            tc, v = flows[0]._native.variants() if flows else (0, 0)
            flows.append(make_flow(_params(_member(c, i, seed), tile_cols=tc, variants=v)))
        nats = [f._native for f in flows]
        states = [_field(_member(c, i, seed), seed + 1000 * i) for i in range(c["members"])]
        nexts = [n.empty() for n in nats]
        plan = BatchPlan(nats, states, nexts, [n.empty() for n in nats], [n.empty() for n in nats], c["slots"])
        return dict(kind=kind, flows=flows, plan=plan, nexts=nexts)
    flow = make_flow(_params(c))
    st = dict(kind=kind, flow=flow, state=_field(c, seed))
    if kind == "run":
        st["steps"] = c["steps"]
    if kind == "guess":
        nat = flow._native
        st.update(mode=c["mode"], hist=_history(c, _rhs(c, st["state"]), seed + 1), pred=nat.empty(),
                  rhs=[nat.empty(), nat.empty()], err=nat.scalar(), net=_mode_net(c, seed) if c["mode"] == 2 else None,
                  walls=c["system"] == "plane-couette")
        if c["mode"] != 4:
            st["hist"] = st["hist"][:2]
    return st


def run(state):
    s = state
    kind = s["kind"]
    if kind == "pgrad":
        loss = s["net"].compute_grad(s["X"], s["T"])
        return dict(grad=s["net"].grad, loss=loss)
    if kind == "pforward":
        return s["net"].forward(s["X"])
    if kind == "mgrad":
        loss = s["net"].compute_grad(s["X"], s["T"], bf16=s["bf16"])
        return dict(grad=s["net"].grad, loss=loss)
    if kind == "ensemble":
        s["plan"].enqueue()
        return s["nexts"]
    flow = s["flow"]
    if kind == "step":
        u = s["state"]
        pred, rhs, _ = flow.predict_and_correct(u)
        pred, rhs, err = flow.iterate_correction(u, pred, rhs)
        pred, _ = flow.correct_velocity(pred)
        return dict(state=pred, rhs=rhs, err=err)
    if kind == "run":
        rec = StatsRecorder(flow, s["state"], it_stats=1)
        res = run_driver(flow, s["state"], s["steps"], callback=rec)
        rec.finish(res.state, len(res.counts))
        return dict(state=res.state, counts=res.counts, energies=rec.Eps)
    nat, h, (ra, rb), mode = flow._native, s["hist"], s["rhs"], s["mode"]
    ops = None if s["net"] is None else s["net"].operands
    cubic = len(h) == 3
    nat.guess(s["state"], s["pred"], ra, h[0], h[1], mode, ops, SCALES, hist3=h[2] if cubic else None,
              carry=not s["walls"])
    s["hist"] = [h[-1]] + h[:-1]  # N^n went to the oldest field
    if s["walls"]:
        nat.iterate_correction(s["state"], s["pred"], ra, rb, s["err"])
        nat.iterate_correction(s["state"], s["pred"], rb, ra, s["err"])
    else:
        nat.iterate_correction_carry(s["pred"], ra, s["err"])
        nat.iterate_correction_carry(s["pred"], ra, s["err"])
    out, _ = flow.correct_velocity(s["pred"])
    return dict(state=out, err=s["err"])


# ---------------------------------------------------------------- work
def _rhs_flops(c):
    """Real-transform arithmetic (5/2 N log2 N) of the six inverse and three
    forward transforms of one nonlinear term, and its pointwise products."""
    px, pz = 3 * c["nx"] // 2, 3 * c["nz"] // 2
    if c["system"] == "plane-couette":
        n, lg = px * c["ny"] * pz, math.log2(px * pz)
    else:
        py = 3 * c["ny"] // 2 if c["oversample_y"] else c["ny"]
        n, lg = px * py * pz, math.log2(px * py * pz)
    return n * (9 * 2.5 * lg + 15)


def work(case):
    c = case
    kind = c["kind"]
    if kind in ("pgrad", "pforward"):
        din, H, dout, B = profile_net.profile_din(c["ny"]), c["hidden"], 6 * c["ny"], c["batch"]
        mults = B * (din * H + H * H + H * dout)
        params = din * H + H * H + H * dout + 2 * H + dout
        if kind == "pforward":
            return dict(bytes=2 * B * din + 4 * B * dout + 4 * params, flops=2 * mults)
        return dict(bytes=2 * B * din + 4 * B * dout + 8 * params, flops=2 * (3 * mults - B * din * H))
    if kind == "mgrad":
        H, B = c["hidden"], c["batch"]
        mults = B * (16 * H + H * H + 6 * H)
        return dict(bytes=4 * B * 22 + 8 * (H * H + 24 * H + 6), flops=2 * (3 * mults - B * 16 * H))
    walls = c["system"] == "plane-couette"
    points = (c["nz"] - 1) * (c["nx"] // 2) * (c["ny"] if walls else c["ny"] - 1)
    S = 48 * points
    flops = _rhs_flops(c)
    if walls:  # two banded solves of four complex right-hand sides in all, and the stencils
        flops += points * (4 * 2 * 2 * 4 * c["p"] + 60 * c["p"])
    if kind == "step":
        return dict(bytes=3 * S, flops=3 * flops)
    if kind == "run":
        return dict(bytes=2 * S, flops=5 * c["steps"] * flops)
    if kind == "guess":
        return dict(bytes=2 * S + (3 if c["mode"] == 4 else 2) * S // 2 + S // 2, flops=3 * flops)
    return dict(bytes=2 * S * c["members"], flops=5 * c["members"] * flops)


# ---------------------------------------------------------------- exact, periodic
def _axis_k(n, length):
    return _harmonics(n, n - 1) * (2 * math.pi / length)


def _grids(c):
    L = 2 * math.pi
    kx = torch.arange(c["nx"] // 2, device=DEV, dtype=F64).view(1, 1, -1) * (2 * math.pi / L)
    return kx, _axis_k(c["ny"], L).view(-1, 1, 1), _axis_k(c["nz"], L).view(1, -1, 1)


def _pad_axis(u, n, P, dim):
    """Stored harmonics of a full axis -> P bins."""
    shape = list(u.shape)
    shape[dim] = P
    out = torch.zeros(shape, dtype=u.dtype, device=u.device)
    h = n // 2
    out.narrow(dim, 0, h).copy_(u.narrow(dim, 0, h))
    out.narrow(dim, P - h + 1, h - 1).copy_(u.narrow(dim, h, h - 1))
    return out


def _cut_axis(u, n, dim):
    P, h = u.shape[dim], n // 2
    return torch.cat([u.narrow(dim, 0, h), u.narrow(dim, P - h + 1, h - 1)], dim)


def _cross(a, b):
    return torch.stack([a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]])


def _periodic_rhs(c, u):
    n, L = (c["ny"], c["nz"], c["nx"]), 2 * math.pi
    P = (3 * n[0] // 2 if c["oversample_y"] else n[0], 3 * n[1] // 2, 3 * n[2] // 2)
    kx, ky, kz = _grids(c)
    k = (kx, ky, kz)
    w = torch.stack([1j * (ky * u[2] - kz * u[1]), 1j * (kz * u[0] - kx * u[2]), 1j * (kx * u[1] - ky * u[0])])

    def phys(v):
        v = _pad_axis(_pad_axis(v, n[0], P[0], 0), n[1], P[1], 1)
        v = torch.fft.ifft(torch.fft.ifft(v, dim=0, norm="forward"), dim=1, norm="forward")
        return torch.fft.irfft(v, n=P[2], dim=2, norm="forward")

    y = torch.arange(P[0], device=DEV, dtype=F64) * (L / P[0])
    kf = 2 * math.pi / L
    U, dU = (torch.sin(kf * y), kf * torch.cos(kf * y)) if c["system"] == "kolmogorov" else (
        torch.cos(kf * y), -kf * torch.sin(kf * y))
    t = math.pi * c["tilt"] / 180.0
    base = [math.cos(t) * U, 0 * U, math.sin(t) * U]
    curl = [math.sin(t) * dU, 0 * U, -math.cos(t) * dU]
    vel = torch.stack([phys(u[i]) + base[i].view(-1, 1, 1) for i in range(3)])
    vort = torch.stack([phys(w[i]) + curl[i].view(-1, 1, 1) for i in range(3)])
    nl = _cross(vel, vort)
    del vel, vort
    s = []
    for i in range(3):
        v = torch.fft.rfft(nl[i], dim=2, norm="forward")[..., : n[2] // 2]
        v = _cut_axis(torch.fft.fft(v, dim=1, norm="forward"), n[1], 1)
        s.append(_cut_axis(torch.fft.fft(v, dim=0, norm="forward"), n[0], 0))
    s = torch.stack(s)
    return _solenoidal(c, s)


def _solenoidal(c, u):
    k = _grids(c)
    k2 = k[0] ** 2 + k[1] ** 2 + k[2] ** 2
    d = (k[0] * u[0] + k[1] * u[1] + k[2] * u[2]) / torch.where(k2 > 0, k2, 1.0)
    return torch.stack([u[i] - k[i] * d for i in range(3)])


def _cn(c):
    """The Crank-Nicolson factors ldt_1 and ildt_2 (zero at the mean mode)."""
    kx, ky, kz = _grids(c)
    k2 = kx**2 + ky**2 + kz**2
    l1 = 1 / c["dt"] - (1 - c["implicitness"]) * k2 / c["re"]
    l2 = 1 / (1 / c["dt"] + c["implicitness"] * k2 / c["re"])
    l1[0, 0, 0] = l2[0, 0, 0] = 0
    return l1, l2


def _periodic_norm(d):
    km = torch.ones(d.shape[-1], device=DEV, dtype=F64) * 2
    km[0] = 1
    return torch.sqrt((km * (d.real**2 + d.imag**2)).sum())


def _mean_zero(c, u):
    u = _solenoidal(c, u)
    u[:, 0, 0, 0] = 0
    return u


# ---------------------------------------------------------------- exact, plane Couette
def _cgl(ny):
    return -torch.cos(torch.arange(ny, device=DEV, dtype=F64) * (math.pi / (ny - 1)))


def _quadrature(y):
    """Weights of the wall-normal integral: Simpson panels on unequal steps;
    with an even number of points the last three intervals take the cubic
    through the last four points."""
    x = y.tolist()
    n = len(x)
    w = [0.0] * n
    m = n if n % 2 else n - 3
    for i in range(0, m - 2, 2):
        h0, h1 = x[i + 1] - x[i], x[i + 2] - x[i + 1]
        s = (h0 + h1) / 6
        w[i] += s * (2 - h1 / h0)
        w[i + 1] += s * (h0 + h1) ** 2 / (h0 * h1)
        w[i + 2] += s * (2 - h0 / h1)
    if n % 2 == 0:
        t = torch.tensor(x[-4:], dtype=F64) - x[-4]
        V = torch.stack([t**j for j in range(4)])
        e = torch.linalg.solve(V, torch.tensor([float(t[3]) ** (j + 1) / (j + 1) for j in range(4)], dtype=F64))
        for j in range(4):
            w[n - 4 + j] += float(e[j])
    return torch.tensor(w, device=DEV, dtype=F64)


def _difference(y, p):
    """D1 on p + 1 and D2 on p + 2 points: each row the derivative of the
    polynomial through its points (a Vandermonde solve in local units)."""
    n = y.numel()
    D = []
    for order, s in ((1, p + 1), (2, p + 2)):
        j0 = [max(0, min(i - s // 2, n - s)) for i in range(n)]
        idx = torch.tensor([[j + q for q in range(s)] for j in j0])
        yc = y.cpu()
        x = yc[idx] - yc[:, None]
        scale = x.abs().amax(1, keepdim=True)
        V = torch.stack([(x / scale) ** q for q in range(s)], 1)
        b = torch.zeros(n, s, 1, dtype=F64)
        b[:, order] = math.factorial(order)
        wts = torch.linalg.solve(V, b)[..., 0] / scale**order
        D.append(torch.zeros(n, n, dtype=F64).scatter_(1, idx, wts).to(DEV))
    return D


def _dy(D, u):
    return torch.complex(u.real @ D.T, u.imag @ D.T)


def _couette_k(c):
    kx = torch.arange(c["nx"] // 2, device=DEV, dtype=F64).view(1, -1, 1)
    return kx, (_harmonics(c["nz"], c["nz"] - 1) * 2.0).view(-1, 1, 1)


def _couette_rhs(c, u, D1):
    nx, nz, ny = c["nx"], c["nz"], c["ny"]
    px, pz = 3 * nx // 2, 3 * nz // 2
    kx, kz = _couette_k(c)
    w = torch.stack([_dy(D1, u[2]) - 1j * kz * u[1], 1j * kz * u[0] - 1j * kx * u[2], 1j * kx * u[1] - _dy(D1, u[0])])

    def phys(v):  # (kz, kx, y) -> (z, x, y)
        v = torch.fft.ifft(_pad_axis(v, nz, pz, 0), dim=0, norm="forward")
        return torch.fft.irfft(v, n=px, dim=1, norm="forward")

    y = _cgl(ny)
    vel = torch.stack([phys(u[i]) for i in range(3)])
    vort = torch.stack([phys(w[i]) for i in range(3)])
    vel[0] += y
    vort[2] -= 1.0
    nl = _cross(vel, vort)
    out = []
    for i in range(3):
        v = torch.fft.rfft(nl[i], dim=1, norm="forward")[:, : nx // 2]
        out.append(_cut_axis(torch.fft.fft(v, dim=0, norm="forward"), nz, 0))
    return torch.stack(out)


class _Influence:
    """The influence-matrix step with dense solves, one factor per k^2."""

    def __init__(self, c):
        self.c = c
        ny, dt, th, nu = c["ny"], c["dt"], c["implicitness"], 1.0 / c["re"]
        self.D1, self.D2 = _difference(_cgl(ny), c["p"])
        self.kx, self.kz = _couette_k(c)
        self.k2 = self.kx**2 + self.kz**2
        k2, self.cls = torch.unique(self.k2.reshape(-1), return_inverse=True)
        self.order = torch.argsort(self.cls, stable=True)
        eye = torch.eye(ny, device=DEV, dtype=F64)
        lap = self.D2 - k2.view(-1, 1, 1) * eye
        H = eye / dt - th * nu * lap
        H[:, 0], H[:, -1] = eye[0], eye[-1]
        L = lap
        L[:, 0], L[:, -1] = self.D1[0], self.D1[-1]
        L[k2 == 0, 0] = eye[0]
        self.L, self.H = self._inverse(L), self._inverse(H)
        self.Lm, self.Hm = L, H
        e = torch.zeros(2, ny, device=DEV, dtype=F64)
        e[0, 0] = e[1, -1] = 1
        P = self._refined(self.L, L, e.T.expand(len(k2), ny, 2))
        r, q = -(self.D1 @ P), P.clone()
        r[:, 0] = r[:, -1] = q[:, 0] = q[:, -1] = 0
        V, Q = self._refined(self.H, H, r), self._refined(self.H, H, q)
        M = torch.stack([self.D1[0] @ V, self.D1[-1] @ V], 1)
        adj = torch.stack([M[:, 1, 1], -M[:, 0, 1], -M[:, 1, 0], M[:, 0, 0]], -1).view(-1, 2, 2)
        inv = adj / (M[:, 0, 0] * M[:, 1, 1] - M[:, 0, 1] * M[:, 1, 0]).view(-1, 1, 1)
        inv[k2 == 0] = 0
        inv[k2 == 0, 1, 1] = 1 / M[k2 == 0, 1, 1]
        self.V, self.Q, self.M = V[self.cls], Q[self.cls], inv[self.cls]

    @staticmethod
    def _inverse(A):
        """Gauss-Jordan with partial pivoting, all matrices side by side."""
        U, n = A.shape[:2]
        B = torch.cat([A, torch.eye(n, device=DEV, dtype=F64).expand(U, n, n)], 2)
        at = torch.arange(U, device=DEV)
        for j in range(n):
            piv = B[:, j:, j].abs().argmax(1) + j
            row = B[at, piv]
            B[at, piv] = B[:, j]
            row = row / row[:, j:j + 1]
            col = B[:, :, j].clone()
            col[:, j] = 0
            B[:, j] = row
            B.baddbmm_(col[:, :, None], row[:, None], alpha=-1)
        return B[:, :, n:].contiguous()

    @staticmethod
    def _refined(inv, A, b):
        """A x = b by the inverse, with two steps of iterative refinement."""
        x = inv @ b
        for _ in range(2):
            x = x + inv @ (b - A @ x)
        return x

    def _solve(self, which, rhs):
        """Per-mode solves of (k, kz, kx, y) complex right-hand sides."""
        inv, A = (self.L, self.Lm) if which == "L" else (self.H, self.Hm)
        n, ny = rhs.shape[0], rhs.shape[-1]
        b = torch.view_as_real(rhs).reshape(n, -1, ny, 2).permute(1, 2, 0, 3).reshape(-1, ny, 2 * n)
        x = torch.empty_like(b)
        step = max(1, (1 << 27) // (ny * ny))
        for i in range(0, b.shape[0], step):
            at = self.order[i:i + step]
            x[at] = self._refined(inv[self.cls[at]], A[self.cls[at]], b[at])
        x = x.reshape(-1, ny, n, 2).permute(2, 0, 1, 3).contiguous()
        return torch.view_as_complex(x).reshape(rhs.shape)

    def step(self, un, uj, nn, nj):
        c = self.c
        dt, th, nu, kx, kz, k2 = c["dt"], c["implicitness"], 1.0 / c["re"], self.kx, self.kz, self.k2
        D1, D2 = self.D1, self.D2

        def div(v):
            return 1j * kx * v[0] + _dy(D1, v[1]) + 1j * kz * v[2]

        d = div(un)
        f = d / dt + th * div(nj) + (1 - th) * div(nn) + (1 - th) * nu * (_dy(D2, d) - k2 * d)
        f[..., 0] = f[..., -1] = 0
        p = self._solve("L", f[None])[0]
        grad = torch.stack([1j * kx * p, _dy(D1, p), 1j * kz * p])
        R = un / dt + (1 - th) * nu * (_dy(D2, un) - k2 * un) - grad + th * nj + (1 - th) * nn
        R[..., 0] = R[..., -1] = 0
        u = self._solve("H", R)
        wall = torch.stack([u[1] @ D1[0].to(C128), u[1] @ D1[-1].to(C128)], -1)
        wall[..., 0] = torch.where(k2[..., 0] == 0, 0, wall[..., 0])
        shape = wall.shape[:2]
        a = -(self.M.to(C128) @ wall.reshape(-1, 2, 1))
        v = (self.V.to(C128) @ a).reshape(*shape, -1)
        q = (self.Q.to(C128) @ a).reshape(*shape, -1)
        new = torch.stack([u[0] - 1j * kx * q, u[1] + v, u[2] - 1j * kz * q])
        return new, new - uj

    def norm(self, d):
        km = torch.where(self.kx == 0, 1.0, 2.0)
        prof = (km * (d.real**2 + d.imag**2)).sum((0, 1, 2))
        return torch.sqrt((prof * _quadrature(_cgl(self.c["ny"]))).sum() / 2.0)


def _rhs(c, u):
    if c["system"] == "plane-couette":
        return _couette_rhs(c, u, _difference(_cgl(c["ny"]), c["p"])[0])
    return _periodic_rhs(c, u)


# ---------------------------------------------------------------- exact
def _layers(net):
    return [w.double() for w in net.unpack()]


def _silu(z):
    return z * torch.sigmoid(z)


def _forward(w, X):
    z1 = X @ w[0] + w[1]
    z2 = _silu(z1) @ w[2] + w[3]
    return _silu(z2) @ w[4] + w[5]


def _exact_net(c, seed):
    X, T = _net_inputs(c, seed)
    net = learned.Net(c["hidden"], seed=seed) if c["kind"] == "mgrad" else profile_net.ProfileNet(
        c["ny"], c["hidden"], seed=seed)
    _some_biases(net, seed)
    w = [x.requires_grad_() for x in _layers(net)]
    if c["kind"] == "pforward":
        with torch.no_grad():
            return _forward(w, X.double())
    d2 = (_forward(w, X.double()) - T.double()) ** 2
    loss = d2.sum(1).mean() if c["kind"] == "mgrad" else d2.mean()
    grads = torch.autograd.grad(loss, w)
    return dict(grad=torch.cat([g.reshape(-1) for g in grads]), loss=loss.detach())


def _exact_run(c, u, steps, tol, max_it):
    """The time loop with the corrector iterated to tolerance."""
    l1, l2 = _cn(c)
    th = c["implicitness"]

    def energy(v):
        return float(_periodic_norm(v)) ** 2 / 2

    energies, counts = [energy(u)], []
    for it in range(steps):
        n0 = _periodic_rhs(c, u)
        v = (u * l1 + n0) * l2
        err, passes = math.inf, 0
        while err > tol and passes <= max_it:
            n1 = _periodic_rhs(c, v)
            d = th * (n1 - n0) * l2
            v, n0, err, passes = v + d, n1, float(_periodic_norm(d)), passes + 1
        u = _mean_zero(c, v)
        counts.append(passes - 1)
        if it + 1 < steps or steps > 1:
            energies.append(energy(u))
    return u, counts, energies


def exact(case, seed):
    c = case
    kind = c["kind"]
    if kind in ("pgrad", "pforward", "mgrad"):
        return _exact_net(c, seed)
    if kind == "ensemble":
        return [_exact_run(_member(c, i, seed), _field(_member(c, i, seed), seed + 1000 * i), 1, 1e-10, 10)[0]
                for i in range(c["members"])]
    u = _field(c, seed)
    if kind == "run":
        state, counts, energies = _exact_run(c, u, c["steps"], 1e-10, 10)
        return dict(state=state, counts=counts, energies=energies)
    walls = c["system"] == "plane-couette"
    n0 = _rhs(c, u)
    if kind == "guess":
        h = [torch.view_as_complex(x.double()) for x in _history(c, n0, seed + 1)]
        d1, d2 = n0 - h[0], n0 - 2 * h[0] + h[1]
        dn = d1 if c["mode"] == 1 else d1 + d2
        if c["mode"] == 4:
            dn = dn + (n0 - 3 * h[0] + 3 * h[1] - h[2])
        if c["mode"] == 2:
            dn = dn + _residual(c, _layers(_mode_net(c, seed)), d1, d2)
    if walls:
        imm = _Influence(c)
        if kind == "guess":
            prev = n0 + dn
            v, _ = imm.step(u, u, prev, prev)
        else:
            prev = n0
            v, _ = imm.step(u, u, n0, n0)
        for _ in range(2):
            new = _couette_rhs(c, v, imm.D1)
            v, d = imm.step(u, v, prev, new)
            prev = new
        return dict(state=v, err=imm.norm(d)) if kind == "guess" else dict(state=v, rhs=prev, err=imm.norm(d))
    l1, l2 = _cn(c)
    th = c["implicitness"]
    v = (u * l1 + n0) * l2
    base = (u * l1 + (1 - th) * n0) * l2
    if kind == "guess":
        v = v + th * l2 * _solenoidal(c, dn)
    for _ in range(2):
        n1 = _periodic_rhs(c, v)
        new = base + th * l2 * n1
        v, d = new, new - v
    state = _mean_zero(c, v)
    return dict(state=state, err=_periodic_norm(d)) if kind == "guess" else dict(state=state, rhs=n1, err=_periodic_norm(d))


def _residual(c, w, d1, d2):
    """The per-point network's estimate of the extrapolation's residual."""
    s1, s2, so = SCALES
    kx, kz = _couette_k(c)
    shape = d1.shape[1:]
    k2 = kx**2 + kz**2
    kmax = max(c["nx"] / 2, 2.0 * (c["nz"] / 2))
    rest = [(c["dt"] * k2 / c["re"]).clamp(max=8.0), kx / kmax, _cgl(c["ny"]), kz / kmax]
    feats = [t for v, s in ((d1, s1), (d2, s2)) for q in range(3) for t in (v[q].real * s, v[q].imag * s)]
    X = torch.stack([f.expand(shape).reshape(-1) for f in feats + rest], 1)
    out = _forward(w, X).reshape(*shape, 6) * so * (1 + c["dt"] * c["implicitness"] * k2 / c["re"])[..., None]
    return torch.stack([torch.complex(out[..., 2 * q], out[..., 2 * q + 1]) for q in range(3)])
