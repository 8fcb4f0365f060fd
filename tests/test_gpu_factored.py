"""The split-precision spectrum on linear omega grids (matrix products over the
steps, synchrad_amd/csrc/factored.h) against the CPU FP64 oracle, at the sizes
where it can go wrong: omega counts around the 32-omega groups and the 128-,
256- and 512-omega tiles, step counts around the 63-step stretches and the
32-step products, every order of the omegas (descending, negative, through
zero), steps that keep part of the frequencies (far and near), and tracks whose amplitude jumps or vanishes.

Bound, per complex field component: each term A_s e^{i phase} passes through at
most eleven FP32-level roundings (two phasor factors and their product on each
side, the amplitude, two fp16 two-word splits of 2^-22 and the dropped low-low
product of 2^-22), at most 11 * 2^-22 = 2.6e-6 of |A_s| in all, and the FP32
accumulation of up to 256 steps (24 additions of 2^-24 of the partial sum) adds
1.4e-6 of the sum of |A_s|: 4e-6 of it together.
"""
from dataclasses import replace

import numpy as np
import pytest
import torch

from oracle import oracle
from synchrad_amd import engine, workloads

pytestmark = pytest.mark.gpu

BOUND = 4e-6


def _far_abs_sum(track, axes, dt):
    """dt * sum_s |A_s| per direction, (n_theta, n_phi), from the reference's definition."""
    x, y, z, ux, uy, uz = track[:6]
    b = np.stack([ux, uy, uz], 1) / np.sqrt(1 + ux ** 2 + uy ** 2 + uz ** 2)[:, None]
    a, m = np.diff(b, axis=0) / dt, 0.5 * (b[1:] + b[:-1])
    out = np.zeros((axes["theta"].size, axes["phi"].size))
    for i, th in enumerate(axes["theta"]):
        for j, ph in enumerate(axes["phi"]):
            n = np.array([np.sin(th) * np.cos(ph), np.sin(th) * np.sin(ph), np.cos(th)])
            c2 = 1 / (1 - m @ n)
            c1 = (a @ n) * c2 ** 2
            out[i, j] = dt * np.linalg.norm(c1[:, None] * (n - m) - c2[:, None] * a, axis=1).sum()
    return out


def _run(mode, comp, tracks, axes, dt, tuning=None, L_screen=None, **kw):
    batch = engine.DeviceBatch(engine.pack_tracks(tracks, dt=dt, **kw))
    ax1 = axes["theta"] if mode == "far" else axes["radius"]
    grid = engine.DeviceGrid(mode, axes["omega"], ax1, axes["phi"], L_screen=L_screen)
    assert grid.omega_step != 0.0
    tuning = replace(tuning or engine.Tuning(), sweep="recurrence")   # short tracks too
    outs = engine.spectrum(batch, grid, comp=comp, precision="float", tuning=tuning)
    torch.cuda.synchronize()
    return {k: o.cpu().numpy().swapaxes(-1, -3) for k, o in zip(engine.COMP_KEYS[comp], outs)}


def _omegas(kind, n):
    lo, hi = 1.0 * workloads.KEV_PER_INV_M, 75.0 * workloads.KEV_PER_INV_M
    return {"up": np.linspace(lo, hi, n), "down": np.linspace(hi, lo, n), "negative": np.linspace(-hi, -lo, n),
            "cross": np.linspace(-0.4 * hi, hi, n), "cross down": np.linspace(0.6 * hi, -hi, n)}[kind]


CASES = [("up", n, 200, 0, 0) for n in (2, 31, 33, 127, 128, 129, 256, 300, 512, 513, 700)] + \
        [("up", 96, n, 0, w) for n, w in ((2, 1), (33, 1), (63, 1), (64, 2), (65, 4), (127, 2), (700, 4))] + \
        [(kind, n, 300, m, 0) for kind, n, m in (("down", 200, 0), ("negative", 150, 2), ("cross", 257, 0),
                                                  ("cross down", 520, 4))]


@pytest.mark.parametrize("kind,n_omega,n_steps,M,W", CASES)
def test_far_edges(kind, n_omega, n_steps, M, W):
    wl = workloads.config2(n_particles=1, n_steps=n_steps, grid=(8, 4, 3))
    axes = dict(wl.axes, omega=_omegas(kind, n_omega))
    tr, dt = wl.track_list(), wl.batch.dt
    ref = oracle.spectrum("far", "cartesian_complex", tr, axes, dt)
    got = _run("far", "cartesian_complex", tr, axes, dt, engine.Tuning(omega_per_lane=M, waves_per_block=W))
    scale = _far_abs_sum(tr[0], axes, dt)[None, None]
    worst = max(float(np.max(np.abs(got[k] - ref[k]) / scale)) for k in ref)
    print(f"{kind} {n_omega} omegas {n_steps} steps M={M} W={W}: {worst:.2e} of sum |A|", flush=True)
    assert worst <= BOUND


def _check_near(wl, tr, axes, dt, tuning=None):
    """The complex field within BOUND of sum_s |v2| + |omega| |v1| at each screen point."""
    L = wl.L_screen
    ref = oracle.spectrum("near", "cartesian_complex", tr, axes, dt, L_screen=L)
    got = _run("near", "cartesian_complex", tr, axes, dt, tuning, L_screen=L)
    x, y, z, ux, uy, uz = tr[0][:6]
    b = (np.stack([ux, uy, uz], 1) / np.sqrt(1 + ux ** 2 + uy ** 2 + uz ** 2)[:, None])[:-1]
    om = np.abs(2 * np.pi * axes["omega"])
    worst = 0.0
    for i, r in enumerate(axes["radius"]):
        for j, ph in enumerate(axes["phi"]):
            d = np.array([r * np.cos(ph), r * np.sin(ph), L]) - np.stack([x, y, z], 1)[:-1]
            R = np.linalg.norm(d, axis=1)
            n = d / R[:, None]
            total = dt * ((1 / R ** 2).sum() + om * (np.linalg.norm(b - n, axis=1) / R).sum())
            worst = max(worst, *(float(np.max(np.abs(got[k] - ref[k])[0, :, i, j] / total)) for k in ref))
    print(f"{axes['omega'].size} omegas {x.size} steps: {worst:.2e} of the sum of the terms", flush=True)
    assert worst <= BOUND


@pytest.mark.parametrize("n_omega,n_steps", [(64, 65), (130, 500), (300, 127)])
def test_near_edges(n_omega, n_steps):
    """Grids that every step keeps whole (past the first, which keeps none)."""
    wl = workloads.config4(n_particles=1)
    tr = [[c[:n_steps] for c in wl.track_list()[0][:6]] + [1.0, 0]]
    axes = {"omega": np.linspace(wl.axes["omega"][0], wl.axes["omega"][-1], n_omega),
            "radius": np.linspace(0.0, 0.07, 3), "phi": np.array([0.0, 2.0])}
    _check_near(wl, tr, axes, wl.batch.dt)


def _near_kept(wl, tr, axes, dt):
    """How many frequencies each step keeps at each screen point, those of smallest |omega|."""
    x, y, z = tr[0][:3]
    om = np.sort(np.abs(axes["omega"]))
    kept = []
    for r in axes["radius"]:
        for ph in axes["phi"]:
            R = np.sqrt((r * np.cos(ph) - x) ** 2 + (r * np.sin(ph) - y) ** 2 + (wl.L_screen - z) ** 2)
            tau = np.arange(x.size) * dt + R
            kept.append(np.searchsorted(om, 0.5 / np.abs(np.diff(tau[:-1]))))
    return np.concatenate(kept)


@pytest.mark.parametrize("kind,n_omega,n_steps,every,M,W", [
    ("up", 31, 300, 1, 0, 1), ("up", 33, 300, 1, 0, 2), ("up", 64, 500, 1, 0, 4), ("up", 65, 500, 3, 2, 1),
    ("up", 129, 700, 1, 0, 0), ("up", 300, 400, 3, 4, 2), ("down", 33, 300, 3, 0, 1), ("down", 129, 700, 1, 0, 4),
    ("negative", 100, 400, 1, 2, 2), ("cross", 65, 500, 1, 0, 0), ("cross down", 260, 500, 3, 0, 1)])
def test_near_cut_steps(kind, n_omega, n_steps, every, M, W):
    """Frequencies across the steps' thresholds, in every order of the grid: steps that
    keep part of a group, in its lower and in its upper half."""
    wl = workloads.config4(n_particles=1)
    dt = every * wl.batch.dt
    tr = [[c[::every][:n_steps] for c in wl.track_list()[0][:6]] + [1.0, 0]]
    lo, hi = wl.axes["omega"][0], 7.3 * wl.axes["omega"][-1]
    omega = {"up": np.linspace(lo, hi, n_omega), "down": np.linspace(hi, lo, n_omega),
             "negative": np.linspace(-hi, -lo, n_omega), "cross": np.linspace(-0.37 * hi, hi, n_omega),
             "cross down": np.linspace(0.61 * hi, -hi, n_omega)}[kind]
    axes = {"omega": omega, "radius": np.linspace(0.0, 0.071, 3), "phi": np.array([0.3, 2.1])}
    if not kind.startswith("cross"):
        kept = _near_kept(wl, tr, axes, dt)
        part = kept[(kept > 0) & (kept < n_omega)] % 32
        assert ((part > 0) & (part <= 16)).sum() > 20 and (part > 16).sum() > 20
    _check_near(wl, tr, axes, dt, engine.Tuning(omega_per_lane=M, waves_per_block=W))


def test_amplitude_range_and_snapshots():
    """An amplitude that is zero for most of the track, tiny, then 1e6 times
    larger: the scale of the fp16 words follows it, and the snapshots taken
    before and after keep their own accuracy (relative to the sum so far)."""
    n, dt = 600, 2e-4
    s = np.arange(n) * dt
    kick = np.where(np.arange(n) < 200, 0.0, np.where(np.arange(n) < 400, 1e-6, 1.0))
    ux = kick * np.sin(40 * s)
    gamma = 30.0
    uz = np.sqrt(gamma ** 2 - 1 - ux ** 2)
    x = np.cumsum(ux / gamma) * dt
    z = np.cumsum(uz / gamma) * dt
    tr = [[x, np.zeros(n), z, ux, np.zeros(n), uz, 1.0, 0]]
    axes = {"omega": np.linspace(10.0, 800.0, 100), "theta": np.linspace(0.0, 0.03, 3), "phi": np.array([0.3, 2.0])}
    ref = oracle.spectrum("far", "cartesian_complex", tr, axes, dt, it_range=(0, n), nSnaps=3)
    got = _run("far", "cartesian_complex", tr, axes, dt, it_range=(0, n), nSnaps=3)
    for snap, end in enumerate((200, 400, 600)):
        scale = _far_abs_sum([c[:end] for c in tr[0][:6]], axes, dt)[None] + 1e-300
        for k in ref:
            assert np.isfinite(got[k]).all()
            assert np.max(np.abs(got[k][snap] - ref[k][snap]) / scale) <= BOUND, (k, snap)


def test_small_component_keeps_its_accuracy():
    """A vertical motion 1e-7 of the horizontal one: each amplitude word has its
    own scale, so the phi component is as accurate, relative to its own sum, as
    the theta component (one common scale would leave it 1e-3 off)."""
    wl = workloads.config1()
    x, y, z, ux, uy, uz = wl.track_list()[0][:6]
    n, dt = 700, wl.batch.dt
    uy = 1e-7 * np.roll(ux, 9)
    y = np.cumsum(uy / 100.0) * dt
    tr = [[c[:n] for c in (x, y, z, ux, uy, uz)] + [1.0, 0]]
    axes = dict(wl.axes, omega=np.linspace(wl.axes["omega"][0], wl.axes["omega"][-1], 100),
                theta=np.linspace(0.0, 0.01, 3), phi=np.array([0.0]))
    ref = oracle.spectrum("far", "spheric_complex", tr, axes, dt)
    got = _run("far", "spheric_complex", tr, axes, dt)
    for pair in (("thetare", "thetaim"), ("phire", "phiim")):
        err = np.sqrt(sum(np.sum((got[k] - ref[k]) ** 2) for k in pair))
        size = np.sqrt(sum(np.sum(ref[k] ** 2) for k in pair))
        print(f"{pair[0][:-2]}: size {size:.2e} rel-L2 {err / size:.2e}", flush=True)
        # BOUND is relative to sum |A_s|; on the undulator line the sum itself is
        # at least a tenth of it in the 2-norm over these omegas
        assert err <= 10 * BOUND * size


@pytest.mark.parametrize("n_steps", [1007, 1008, 1009])
@pytest.mark.parametrize("kind,n_omega", [("up", 2), ("up", 24), ("down", 33), ("cross", 64)])
def test_small_grids_of_long_tracks(kind, n_omega, n_steps):
    """Grids of at most one wave's frequencies, at the track length from which they take
    the factored tiles by themselves; four waves share the steps."""
    test_far_edges(kind, n_omega, n_steps, 0, 0)


@pytest.mark.parametrize("n_steps", [64, 95, 96, 126, 127, 158, 190, 253])
@pytest.mark.parametrize("n_omega", [100, 200, 400])
def test_blocks_in_succession(n_omega, n_steps):
    """One wave sweeping one, two and three blocks of steps with nothing between them:
    two blocks of one queue, and at the track's end the rest of every queue, each
    rewriting the factors that the block before has read."""
    test_far_edges("up", n_omega, n_steps, 0, 1)
