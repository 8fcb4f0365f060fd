"""The FP64 tile kernel's groups of threads that share a tile's steps (launches
short of waves) against the CPU FP64 oracle: track lengths around the parts'
and the staged tiles' edges, several snapshots, both field modes, and a batch
large enough not to need them.

FP64 bar of the path: 1e-10 relative L2 (the parts only regroup the FP64 sums,
~1e-15)."""
import numpy as np
import pytest

from oracle import oracle
from synchrad_amd import engine, workloads
from test_gpu_parity import F64_TOL, check, gpu_spectrum

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_omega", [5, 64, 130])
@pytest.mark.parametrize("n_steps", [2, 127, 128, 129, 257, 1000, 2049])
def test_far_parts(n_omega, n_steps):
    wl = workloads.config2(n_particles=1, n_steps=n_steps, grid=(n_omega, 4, 3))
    tr = wl.track_list()
    ref = oracle.spectrum("far", "cartesian", tr, wl.axes, wl.batch.dt)
    got = gpu_spectrum(tr, wl.axes, wl.batch.dt, comp="cartesian")
    # against the norm of all three: on the axis z holds rounding residue only
    err = np.sqrt(sum(np.sum((got[k] - ref[k]) ** 2) for k in ref) / sum(np.sum(ref[k] ** 2) for k in ref))
    print(f"{n_omega} x {n_steps}: rel-L2 {err:.3e}", flush=True)
    assert err <= F64_TOL


@pytest.mark.parametrize("it_range,nSnaps", [(None, 3), ((0, 1500), 4)])
def test_parts_and_snapshots(it_range, nSnaps):
    """Records inside a track: the groups' sums meet at each and go on from there."""
    wl = workloads.config2(n_particles=2, n_steps=1400, grid=(40, 3, 3))
    tr = [[c[:n] for c in t[:6]] + [t[6], 0] for t, n in zip(wl.track_list(), (1400, 901))]
    ref = oracle.spectrum("far", "cartesian_complex", tr, wl.axes, wl.batch.dt, it_range=it_range, nSnaps=nSnaps)
    got = gpu_spectrum(tr, wl.axes, wl.batch.dt, comp="cartesian_complex", it_range=it_range, nSnaps=nSnaps)
    check(got, ref, "double", f"snapshots {it_range}")


@pytest.mark.parametrize("precision,W", [("double", 0), ("double", 4), ("float", 1), ("float", 4)])
@pytest.mark.parametrize("it_range,nSnaps", [((0, 1500), 11), ((0, 1500), 60), ((0, 1500), 375), ((200, 900), 700), (None, 300)])
def test_many_records(precision, W, it_range, nSnaps):
    """Records at every distance, down to one at each step: parts of the steps between
    records, and records inside a staged tile, on its last step and after the last active
    one (FP64, and the split direct sweep on a logarithmic grid)."""
    wl = workloads.config2(n_particles=2, n_steps=1400, grid=(40, 3, 2))
    axes = dict(wl.axes)
    if precision == "float":
        axes["omega"] = np.geomspace(axes["omega"][0], axes["omega"][-1], 40)
    tr = [[c[:n] for c in t[:6]] + [t[6], its] for t, n, its in zip(wl.track_list(), (1400, 301), (0, 150))]
    ref = oracle.spectrum("far", "total", tr, axes, wl.batch.dt, it_range=it_range, nSnaps=nSnaps)
    got = gpu_spectrum(tr, axes, wl.batch.dt, precision=precision, it_range=it_range, nSnaps=nSnaps,
                       tuning=engine.Tuning(waves_per_block=W))
    check(got, ref, precision, f"{nSnaps} records")


@pytest.mark.parametrize("nSnaps", [7, 40, 350])
def test_near_many_records(nSnaps):
    wl = workloads.config4(n_particles=1)
    tr = [[c[:700] for c in wl.track_list()[0][:6]] + [1.0, 0]]
    axes = dict(omega=wl.axes["omega"][:70], radius=wl.axes["radius"][::24], phi=wl.axes["phi"][::32])
    ref = oracle.spectrum("near", "cartesian_complex", tr, axes, wl.batch.dt, L_screen=wl.L_screen, nSnaps=nSnaps)
    got = gpu_spectrum(tr, axes, wl.batch.dt, mode="near", comp="cartesian_complex", L_screen=wl.L_screen, nSnaps=nSnaps)
    check(got, ref, "double", f"near {nSnaps} records")


@pytest.mark.parametrize("n_steps", [700, 2300])
def test_near_parts(n_steps):
    """The longer track takes the largest block, 16 waves: its LDS is past 64 KiB."""
    wl = workloads.config4(n_particles=1)
    tr = [[c[:n_steps] for c in wl.track_list()[0][:6]] + [1.0, 0]]
    axes = dict(omega=wl.axes["omega"], radius=wl.axes["radius"][::16], phi=wl.axes["phi"][::16])
    ref = oracle.spectrum("near", "total", tr, axes, wl.batch.dt, L_screen=wl.L_screen)
    got = gpu_spectrum(tr, axes, wl.batch.dt, mode="near", L_screen=wl.L_screen)
    check(got, ref, "double", "near")


def test_explicit_shapes_keep_their_results():
    """Every block shape, with the parts its waves leave room for."""
    wl = workloads.config2(n_particles=1, n_steps=1100, grid=(70, 4, 2))
    tr = wl.track_list()
    ref = oracle.spectrum("far", "total", tr, wl.axes, wl.batch.dt)
    for m in (1, 2):
        for w in (1, 2, 4):
            got = gpu_spectrum(tr, wl.axes, wl.batch.dt, tuning=engine.Tuning(omega_per_lane=m, waves_per_block=w))
            check(got, ref, "double", f"M={m} W={w}")
            assert np.all(got["total"] >= 0)
