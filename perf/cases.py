"""What users of this framework have it do, as cases that can be timed and checked.

A case is one spectrum (or one spectrum with its gradients) of a set of electron
tracks.  The tracks are those of the workloads module -- a betatron beam in a
plasma channel, planar and helical undulator orbits -- made here on the GPU from
a seed, with the momenta at t_i and the positions half a step later in the far
field, as the calculator's own examples lay them out.

    listed()            the cases
    draw(rng)           one more of the same ranges
    prepare(case, seed) tracks, grid and calculator in hand before the call
    run(state)          one pass through the public entry points
    work(case)          bytes and operations of one pass
    tolerance(case)     how far another correct implementation may be off
    exact(case, seed)   the same outputs in plain 64-bit torch, or None

The sizes: the undulator of 1600 steps on 256 x 32 x 32 and its 32 x 4 x 4
reduction, the betatron beam of 8000 steps on 512 x 64 x 64, the uneven batch on
a logarithmic grid, the near-field screens and the adjoint workload of 128 x 32 x
32 are the configurations of ``synchrad_amd.workloads``; particle counts are cut
so that a pass stays under a second.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from synchrad_amd import autograd, calc, engine, workloads

DEVICE = "cuda"
TWO_PI = 2.0 * math.pi


def listed():
    base = dict(call="spectrum", mode="far", comp="total", precision="float", axis="linear", snaps=1,
                window=False, ragged=False, sigma=0.0)

    def case(name, **kw):
        return dict(base, name=name, **kw)

    return [
        # the smallest call a program makes, e.g. once per optimisation step on a
        # few directions: latency and launches
        case("tiny-double", beam="undulator", precision="double", particles=1, steps=1600,
             n_omega=32, n_axis=4, n_phi=4),
        # the drop-in calculator on host tracks, one electron, default precision:
        # upload, spectrum, axis swap and download
        case("calculator-double", call="calculator", beam="undulator", precision="double", particles=1,
             steps=1600, n_omega=256, n_axis=32, n_phi=32),
        # the same undulator line resident on the GPU in single precision
        case("undulator-float", beam="undulator", particles=1, steps=1600,
             n_omega=256, n_axis=32, n_phi=32),
        # a small betatron beam, the usual exploratory run, in both precisions
        case("betatron-float", beam="betatron", particles=24, steps=8000,
             n_omega=512, n_axis=32, n_phi=32),
        case("betatron-double", beam="betatron", precision="double", particles=24, steps=4000,
             n_omega=256, n_axis=32, n_phi=32),
        # a tenth of the production betatron beam on its full grid
        case("betatron-large", beam="betatron", particles=200, steps=8000,
             n_omega=512, n_axis=64, n_phi=64),
        # uneven track lengths, logarithmic frequencies, three components
        case("uneven-log", beam="mixed", comp="cartesian", axis="log", ragged=True, particles=120, steps=20000,
             n_omega=256, n_axis=32, n_phi=32),
        # coherent amplitudes at several snapshots of one global time window, odd sizes
        case("snapshots-complex", beam="mixed", comp="cartesian_complex", window=True, ragged=True, snaps=3,
             particles=50, steps=2100, n_omega=200, n_axis=15, n_phi=12, sigma=1e-10),
        # near-field screen a few metres behind the undulator
        case("near-float", mode="near", beam="undulator", particles=48, steps=4000,
             n_omega=128, n_axis=64, n_phi=64),
        case("near-double", mode="near", beam="undulator", precision="double", comp="cartesian", particles=2,
             steps=1500, n_omega=100, n_axis=48, n_phi=24),
        # spectrum and gradients of every sample and weight, forward and backward
        case("adjoint-float", call="adjoint", beam="betatron", particles=64, steps=4000,
             n_omega=128, n_axis=32, n_phi=32),
        case("adjoint-double", call="adjoint", beam="betatron", precision="double", particles=8, steps=1500,
             n_omega=100, n_axis=12, n_phi=12),
    ]


def _spread(rng, lo, hi):
    """A whole number in [lo, hi], even over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["far", "far", "far", "log", "window", "near", "adjoint", "calculator"])
    precision = rng.choice(["float", "float", "double"])
    case = dict(call="spectrum", mode="far", comp="total", precision=precision, axis="linear", snaps=1,
                window=False, ragged=False, sigma=0.0, beam=rng.choice(["betatron", "undulator"]))
    grid = [_spread(rng, 24, 1100), _spread(rng, 1, 64), _spread(rng, 1, 64)]
    case["particles"], case["steps"] = _spread(rng, 1, 300), _spread(rng, 150, 8000)
    budget = 4e11 if precision == "float" else 1.2e11
    if kind == "far":
        case["comp"] = rng.choice(["total", "total", "cartesian", "spheric", "spheric_complex"])
    elif kind == "log":
        case.update(beam="mixed", axis=rng.choice(["log", "wavelength"]), ragged=True,
                    comp=rng.choice(["total", "cartesian"]))
    elif kind == "window":
        case.update(beam="mixed", ragged=True, window=True, snaps=rng.randint(1, 5), comp="cartesian_complex",
                    sigma=rng.choice([0.0, 1e-10]))
    elif kind == "near":
        case.update(mode="near", beam="undulator", comp=rng.choice(["total", "cartesian", "cartesian_complex"]))
        budget *= 0.5
    elif kind == "adjoint":
        case.update(call="adjoint", beam="betatron", comp=rng.choice(["total", "cartesian"]))
        grid = [_spread(rng, 24, 600), _spread(rng, 2, 32), _spread(rng, 2, 32)]
        budget *= 0.1
    else:
        case.update(call="calculator")
        case["particles"] = _spread(rng, 1, 20)
        budget *= 0.1
    while case["particles"] * case["steps"] * grid[0] * grid[1] * grid[2] > budget:
        if case["particles"] > 4:
            case["particles"] = (case["particles"] + 1) // 2
        elif grid[1] * grid[2] > 256:
            grid[1], grid[2] = (grid[1] + 1) // 2, (grid[2] + 1) // 2
        else:
            case["steps"] = max(150, case["steps"] // 2)
    case["n_omega"], case["n_axis"], case["n_phi"] = grid
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
UNDULATOR_PERIOD = 0.01


def _shape(case):
    return case["n_omega"], case["n_axis"], case["n_phi"]


def _time_step(case):
    if case["beam"] == "betatron":
        return TWO_PI / (200.0 * workloads.plasma_kp())
    return UNDULATOR_PERIOD / (24 if case["beam"] == "mixed" else 32)


def _axes(case):
    """The calculator's axes (1/lambda, angle or radius, azimuth) as numpy arrays."""
    n_w, n1, n_p = _shape(case)
    if case["beam"] == "betatron":
        lo, hi, top = 1.0 * workloads.KEV_PER_INV_M, 75.0 * workloads.KEV_PER_INV_M, 0.04
    elif case["beam"] == "mixed":
        lo = 0.5 * workloads.undulator_omega1(50.0, 3.0, UNDULATOR_PERIOD)
        hi = 2.0 * workloads.undulator_omega1(500.0, 0.5, UNDULATOR_PERIOD)
        top = 0.06
        if case["axis"] == "linear":
            hi = 0.02 * hi
    else:
        line = workloads.undulator_omega1(100.0, 1.0, UNDULATOR_PERIOD)
        lo, hi, top = 0.5 * line, 1.5 * line, 0.01
    if case["mode"] == "near":
        top = 0.05
    features = {"linear": [], "log": ["logGrid"], "wavelength": ["wavelengthGrid"]}[case["axis"]]
    omega, _ = calc.frequency_nodes(lo, hi, n_w, features)
    return omega, calc.inclusive_nodes(0.0, top, n1), calc.periodic_nodes(0.0, TWO_PI, n_p), (lo, hi, top), features


def _lengths(case, seed):
    rng = np.random.default_rng(7919 + seed)
    n_p, top = case["particles"], case["steps"]
    if not case["ragged"]:
        return np.full(n_p, top, dtype=np.int64)
    return np.round(np.exp(rng.uniform(math.log(max(2, top // 100)), math.log(top), n_p))).astype(np.int64)


def _tracks(case, seed):
    """(offsets, [x, y, z, ux, uy, uz] and weights as GPU float64, it_start, it_range)."""
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    f64 = dict(dtype=torch.float64, device=DEVICE)
    n_p = case["particles"]
    normal = lambda: torch.randn(n_p, generator=gen, **f64)
    uniform = lambda lo, hi: lo + (hi - lo) * torch.rand(n_p, generator=gen, **f64)
    lengths = _lengths(case, seed)
    offsets = np.zeros(n_p + 1, dtype=np.int64)
    np.cumsum(lengths, out=offsets[1:])
    cdt = _time_step(case)
    stagger = 0.5 * cdt if case["mode"] == "far" else 0.0
    which = torch.repeat_interleave(torch.arange(n_p, device=DEVICE), torch.from_numpy(lengths).to(DEVICE))
    step = torch.arange(int(offsets[-1]), device=DEVICE) - torch.from_numpy(offsets[:-1]).to(DEVICE)[which]
    s = step.to(torch.float64) * cdt
    sp = s + stagger
    if case["beam"] == "betatron":
        # harmonic motion in the channel; z is summed from the momenta
        gamma, x0, y0 = 400.0 + 16.0 * normal(), 1e-6 * normal(), 1e-6 * normal()
        ux0, uy0 = 2.0 * normal(), 2.0 * normal()
        kb = workloads.plasma_kp() / torch.sqrt(2.0 * gamma)
        g, k = gamma[which], kb[which]
        ux = ux0[which] * torch.cos(k * s) - g * k * x0[which] * torch.sin(k * s)
        uy = uy0[which] * torch.cos(k * s) - g * k * y0[which] * torch.sin(k * s)
        x = x0[which] * torch.cos(k * sp) + ux0[which] / (g * k) * torch.sin(k * sp)
        y = y0[which] * torch.cos(k * sp) + uy0[which] / (g * k) * torch.sin(k * sp)
        uz = torch.sqrt(g * g - 1.0 - ux * ux - uy * uy)
        z = torch.cumsum((uz / g * cdt).view(n_p, -1), dim=1).reshape(-1)
    else:
        # planar (and, mixed, every other one helical) undulator orbits
        ku = TWO_PI / UNDULATOR_PERIOD
        if case["beam"] == "mixed":
            gamma, K, psi = uniform(50.0, 500.0), uniform(0.5, 3.0), uniform(0.0, TWO_PI)
            helical = (torch.arange(n_p, device=DEVICE) % 2).to(torch.float64)
        else:
            gamma, K, psi = 100.0 * (1.0 + 0.005 * normal()), 1.0 + 0.0 * normal(), 0.0 * normal()
            helical = torch.zeros(n_p, **f64)
        x0, y0 = 20e-6 * normal(), 20e-6 * normal()
        g, kk, ps, he = gamma[which], K[which], psi[which], helical[which]
        a, b = ku * s + ps, ku * sp + ps
        ux = kk * torch.cos(a)
        uy = he * kk * torch.sin(a)
        uz = torch.sqrt(g * g - 1.0 - ux * ux - uy * uy)
        x = x0[which] + kk / (g * ku) * (torch.sin(b) - torch.sin(ps))
        y = y0[which] - he * kk / (g * ku) * (torch.cos(b) - torch.cos(ps))
        bbar = 1.0 - (1.0 + kk * kk * 0.5 * (1.0 + he)) / (2.0 * g * g)
        z = bbar * sp - (1.0 - he) * kk * kk / (8.0 * g * g * ku) * (torch.sin(2.0 * b) - torch.sin(2.0 * ps))
    w = uniform(0.5, 1.5)
    it_start, it_range = None, None
    if case["window"]:
        start = np.random.default_rng(104729 + seed).integers(0, max(1, case["steps"] // 4), n_p)
        it_start, it_range = start.astype(np.uint32), (0, case["steps"])
    cols = [t.contiguous() for t in (x, y, z, ux, uy, uz)]
    return offsets, cols, w, it_start, it_range


def _screen(case):
    """Distance of the near-field screen: behind the end of the track."""
    return case["steps"] * _time_step(case) + 5.0 if case["mode"] == "near" else None


def prepare(case, seed):
    offsets, cols, w, it_start, it_range = _tracks(case, seed)
    omega, ax1, phi, (lo, hi, top), features = _axes(case)
    cdt = _time_step(case)
    host = [c.cpu().numpy() for c in cols]
    if case["call"] == "calculator":
        tracks = [[*(c[a:b].copy() for c in host), float(wp), 0]
                  for a, b, wp in zip(offsets[:-1], offsets[1:], w.cpu().numpy())]
        calculator = calc.SynchRad({"grid": [(lo, hi), (0.0, top), (0.0, TWO_PI), _shape(case)],
                                    "dtype": case["precision"], "mode": case["mode"], "Features": features})
        return dict(case=case, calculator=calculator, tracks=tracks, cdt=cdt)
    packed = engine.pack_csr(offsets, *host, w.cpu().numpy(), it_start, dt=cdt, it_range=it_range,
                             nSnaps=case["snaps"])
    grid = engine.DeviceGrid(case["mode"], omega, ax1, phi, L_screen=_screen(case))
    state = dict(case=case, grid=grid)
    if case["call"] == "adjoint":
        state.update(layout=packed, leaves=[t.clone().requires_grad_(True) for t in (*cols, w)],
                     weight=_upstream(case, seed))
    else:
        state.update(batch=engine.DeviceBatch(packed))
    return state


def _upstream(case, seed):
    """dL/dS: the derivative of the user's loss with respect to the spectra."""
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed + 50021)
    n_w, n1, n_p = _shape(case)
    n_out = 1 if case["comp"] == "total" else 3
    return torch.randn((n_out, 1, n_p, n1, n_w), generator=gen, dtype=torch.float64, device=DEVICE)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    case = state["case"]
    if case["call"] == "calculator":
        c = state["calculator"]
        c.calculate_spectrum(state["tracks"], timeStep=state["cdt"], comp=case["comp"],
                             sigma_particle=case["sigma"], L_screen=_screen(case), verbose=False)
        return [c.Data["radiation"][k] for k in engine.COMP_KEYS[case["comp"]]]
    if case["call"] == "adjoint":
        leaves = state["leaves"]
        S = autograd.far_spectrum(*leaves, state["layout"], state["grid"], comp=case["comp"],
                                  precision=case["precision"])
        grads = torch.autograd.grad(S, leaves, grad_outputs=state["weight"])
        return [S.detach(), *grads]
    return engine.spectrum(state["batch"], state["grid"], comp=case["comp"], precision=case["precision"],
                           sigma_particle=case["sigma"])


def _samples(case):
    """Samples of the tracks (ragged lengths: their expectation, log-uniform)."""
    if not case["ragged"]:
        return case["particles"] * case["steps"]
    top = case["steps"]
    low = max(2, top // 100)
    return case["particles"] * (top - low) / math.log(top / low)


def work(case):
    """Bytes: every sample, weight and (backward) upstream derivative read once,
    every output written once.  Operations: the sum itself, per sample and
    spectral point -- two complex amplitude words in the far field (four
    multiply-adds), six in the near field (twelve), three times that for a
    spectrum with its gradients; forming the phases and amplitudes, which can be
    shared between spectral points, is not counted, and neither is that the
    phase filter leaves part of the pairs out."""
    n = _samples(case)
    points = math.prod(_shape(case))
    n_out = len(engine.COMP_KEYS[case["comp"]])
    bytes_ = 48.0 * n + 8.0 * case["particles"] + 8.0 * n_out * points * case["snaps"]
    flops = n * points * (8.0 if case["mode"] == "far" else 24.0)
    if case["call"] == "adjoint":
        bytes_ = 2.0 * bytes_ + 48.0 * n
        flops *= 3.0
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """Double: the phases reach 1e5 rad and more, so 64-bit rounding of a
    phase moves a term by 1e-11.  Float: 32-bit amplitudes, sines and sums,
    measured 7e-8 to 3e-7 off the 64-bit result; the momentum gradients are
    differences of neighbouring steps' sums, measured 1e-5 to 2.3e-5 off."""
    if case["precision"] == "double":
        return {"rel": 1e-10, "max": 1e-8}
    if case["call"] == "adjoint":
        return {"rel": 1e-4, "max": 4e-3}
    return {"rel": 1.5e-6, "max": 1e-4}


# ---------------------------------------------------------------------------
# the same in plain 64-bit torch
# ---------------------------------------------------------------------------
EXACT_PAIRS = 1.5e11          # about 15 seconds
CHUNK = 1 << 25


def _directions(case):
    """Far: unit vectors (n_phi * n_theta, 3); near: screen points."""
    _, ax1, phi, _, _ = _axes(case)
    if case["mode"] == "far":
        st, ct = np.sin(ax1)[None, :], np.cos(ax1)[None, :]
        sp, cp = np.sin(phi)[:, None], np.cos(phi)[:, None]
        v = np.stack([st * cp, st * sp, np.broadcast_to(ct, (phi.size, ax1.size))], axis=-1)
    else:
        r = ax1[None, :]
        v = np.stack([r * np.cos(phi)[:, None], r * np.sin(phi)[:, None],
                      np.full((phi.size, ax1.size), _screen(case))], axis=-1)
    return torch.from_numpy(v.reshape(-1, 3)).to(DEVICE)


def _spheric(case):
    """e_r, e_theta, e_phi of every direction, (directions, 3, 3)."""
    _, ax1, phi, _, _ = _axes(case)
    t, p = np.meshgrid(ax1, phi)
    st, ct, sp, cp = np.sin(t), np.cos(t), np.sin(p), np.cos(p)
    e = np.stack([np.stack([st * cp, st * sp, ct], -1), np.stack([ct * cp, ct * sp, -st], -1),
                  np.stack([-sp, cp, 0.0 * cp], -1)], axis=-2)
    return torch.from_numpy(e.reshape(-1, 3, 3)).to(DEVICE)


def _parts(case, track, n_steps, its, cdt, omega, dirs, cuts):
    """(re, im) sums over the steps up to each cut: lists of (D, n_w, 3)."""
    x, y, z, ux, uy, uz = (t[:n_steps + 1] for t in track)
    time = (torch.arange(n_steps, device=DEVICE) + its).to(torch.float64) * cdt
    ginv = 1.0 / torch.sqrt(1.0 + (ux * ux + uy * uy + uz * uz))
    b = torch.stack([ux * ginv, uy * ginv, uz * ginv], dim=-1)
    r = torch.stack([x, y, z], dim=-1)[:n_steps]
    if case["mode"] == "far":
        tau = time - (r[:, 0] * dirs[:, 0:1] + r[:, 1] * dirs[:, 1:2] + r[:, 2] * dirs[:, 2:3])
        a, m = (b[1:] - b[:-1]) * (1.0 / cdt), 0.5 * (b[1:] + b[:-1])
        n = dirs[:, None, :]
        c2 = 1.0 / (1.0 - (m[:, 0] * n[..., 0] + m[:, 1] * n[..., 1] + m[:, 2] * n[..., 2]))
        c1 = (a[:, 0] * n[..., 0] + a[:, 1] * n[..., 1] + a[:, 2] * n[..., 2]) * c2 * c2
        amp = c1[..., None] * (n - m) - c2[..., None] * a
    else:
        d = dirs[:, None, :] - r
        dist = torch.sqrt(d[..., 0] ** 2 + d[..., 1] ** 2 + d[..., 2] ** 2)
        tau = time + dist
        n = d / dist[..., None]
        amp = torch.cat([(b[:n_steps] - n) / dist[..., None], n / (dist * dist)[..., None]], dim=-1)
    phase = omega[None, :, None] * tau[:, None, :]
    with torch.no_grad():
        diff = phase.detach().clone()
        diff[..., 1:] -= phase[..., :-1]
        keep = diff.abs() < math.pi
        del diff
    cos, sin = torch.where(keep, torch.cos(phase), 0.0), torch.where(keep, torch.sin(phase), 0.0)
    out, lo, re, im = [], 0, 0.0, 0.0
    for hi in cuts:
        if hi > lo:
            pc = torch.matmul(cos[..., lo:hi], amp[:, lo:hi])
            ps = torch.matmul(sin[..., lo:hi], amp[:, lo:hi])
            if case["mode"] == "near":
                w = omega[None, :, None]
                pc, ps = pc[..., 3:] - w * ps[..., :3], ps[..., 3:] + w * pc[..., :3]
            re, im, lo = re + pc, im + ps, hi
        out.append((re, im))
    return out


def _records(case, n, its, it_range):
    """(slot, number of summed steps) of a particle's snapshot records."""
    last_it = int(it_range[-1]) if it_range is not None else n
    its = its if it_range is not None else 0
    grid = np.linspace(*(it_range if it_range is not None else (0, n)), case["snaps"] + 1, dtype=np.uint32)[1:]
    active = min(n - 1, last_it - 1)
    out, prev, slot = [], -1, 0
    while slot < len(grid) and its >= int(grid[slot]):
        slot += 1
    for k in range(slot, len(grid)):
        r = int(grid[k]) - 2 - its
        if r <= prev or r > last_it - 2:
            break
        out.append((k, max(0, min(r + 1, active))))
        prev = r
    return its, out


def exact(case, seed):
    n_w, n1, n_p = _shape(case)
    if _samples(case) * n_w * n1 * n_p * (3.0 if case["call"] == "adjoint" else 1.0) > EXACT_PAIRS:
        return None
    offsets, cols, weights, it_start, it_range = _tracks(case, seed)
    omega, _, _, _, _ = _axes(case)
    omega_d = torch.from_numpy(np.double(2 * np.pi) * omega).to(DEVICE)
    cdt, dirs = _time_step(case), _directions(case)
    comp, n_dir = case["comp"], dirs.shape[0]
    n_out = len(engine.COMP_KEYS[comp])
    outs = torch.zeros((n_out, case["snaps"], n_dir, n_w), dtype=torch.float64, device=DEVICE)
    backward = case["call"] == "adjoint"
    up = _upstream(case, seed).reshape(n_out, n_dir, n_w) if backward else None
    grads = [torch.zeros_like(c) for c in (*cols, weights)]
    basis = _spheric(case) if comp.startswith("spheric") else None
    factor = torch.ones(n_w, dtype=torch.float64, device=DEVICE)
    if comp == "cartesian_complex" and case["mode"] == "far":
        factor = torch.exp(-0.5 * (omega_d * case["sigma"]) ** 2)
    for p in range(case["particles"]):
        a, b = int(offsets[p]), int(offsets[p + 1])
        its, records = _records(case, b - a, int(it_start[p]) if it_start is not None else 0, it_range)
        steps = max((c for _, c in records), default=0)
        if not records:
            continue
        track = [c[a:b].detach().clone().requires_grad_(backward) for c in cols]
        w = weights[p].detach().clone().requires_grad_(backward)
        per = max(1, CHUNK // max(1, n_w * steps))
        for d0 in range(0, n_dir, per):
            sl = slice(d0, min(n_dir, d0 + per))
            sums = _parts(case, track, steps, its, cdt, omega_d, dirs[sl], [c for _, c in records])
            for (slot, _), (re, im) in zip(records, sums):
                if isinstance(re, float):
                    continue
                if basis is not None:
                    re, im = (torch.matmul(v, basis[sl].transpose(1, 2)) for v in (re, im))
                    if comp == "spheric_complex" or comp == "spheric":
                        # the field is transverse: its radial part is rounding
                        re, im = (torch.cat([0.0 * v[..., :1], v[..., 1:]], dim=-1) for v in (re, im))
                if comp == "total":
                    val = [w * cdt * cdt * (re ** 2 + im ** 2).sum(-1)]
                elif comp in ("cartesian", "spheric"):
                    val = [w * cdt * cdt * (re[..., c] ** 2 + im[..., c] ** 2) for c in range(3)]
                else:
                    val = [torch.sqrt(w) * cdt * factor * v[..., c] for c in range(3) for v in (re, im)]
                for c, v in enumerate(val):
                    outs[c, slot, sl] += v.detach()
                if backward:
                    sum((v * up[c, sl]).sum() for c, v in enumerate(val)).backward()
        if backward:
            for g, t in zip(grads, track):
                g[a:b] += t.grad
            grads[6][p] += w.grad
    outs = outs.reshape(n_out, case["snaps"], n_p, n1, n_w)
    if backward:
        return [outs, *grads]
    if case["call"] == "calculator":
        return [o.transpose(-1, -3).contiguous().cpu().numpy() for o in outs]
    return [o.contiguous() for o in outs]
