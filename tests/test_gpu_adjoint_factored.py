"""The split-precision adjoint on linear omega grids (matrix products over the
frequencies) against the FP64 path, at the sizes where it can go wrong: edges of the
groups of 32 frequencies and of the tiles, of the 64-step waves and the blocks' runs
of steps, direction groups and batches, tracks whose steps cut the frequencies, and
grids that cross zero.

Bar: the sums' words carry 2^-22 of their largest coefficient, the phases' sines
2^-23; gradients of the weights and positions stay below 2e-5 relative L2 and those of
the momenta, differences of neighbouring steps' sums, below the split path's 1e-4."""
import numpy as np
import pytest
import torch

from synchrad_amd import engine, workloads

pytestmark = pytest.mark.gpu

BARS = [2e-5] * 3 + [1e-4] * 3 + [2e-5]


def _grads(hb, grid, G, comp, precision, tuning=None, fields=None):
    out = engine.far_adjoint(engine.DeviceBatch(hb), grid, G, comp=comp, precision=precision, tuning=tuning, fields=fields)
    torch.cuda.synchronize()
    return out


def _check(wl, axes, comp="total", tuning=None, seed=5, it_range=None, tracks=None, exact_fields=False, bars=BARS):
    grid = engine.DeviceGrid("far", axes["omega"], axes["theta"], axes["phi"])
    hb = engine.pack_tracks(tracks or wl.track_list(), dt=wl.batch.dt, it_range=it_range)
    rng = np.random.default_rng(seed)
    shape = (1, axes["phi"].size, axes["theta"].size, axes["omega"].size)
    G = [torch.from_numpy(rng.standard_normal(shape)).cuda() for _ in range(1 if comp == "total" else 3)]
    fields = engine.far_fields(engine.DeviceBatch(hb), grid, comp=comp, precision="double")[0] if exact_fields else None
    got = _grads(hb, grid, G, comp, "float", tuning, fields)
    ref = _grads(hb, grid, G, comp, "double")
    for c in range(7):
        n = float(torch.linalg.norm(ref[c]))
        r = float(torch.linalg.norm(got[c] - ref[c])) / n if n > 0 else 0.0
        print(f"{comp} grad[{c}]: rel-L2 {r:.3e}", flush=True)
        assert r <= bars[c], (c, r)


@pytest.mark.parametrize("comp,n_omega", [("total", n) for n in (24, 31, 32, 33, 64, 65, 129, 257, 512, 513)] +
                         [("cartesian", n) for n in (64, 65, 129, 256, 257, 513)])
def test_group_and_tile_edges(n_omega, comp):
    # tracks long enough for the matrix products: 20000 (step, omega) pairs
    n_steps = max(400, 20000 // n_omega + 1) if comp == "total" else 1050
    wl = workloads.config2(n_particles=2, n_steps=n_steps, grid=(n_omega, 3, 2))
    _check(wl, wl.axes, comp)


@pytest.mark.parametrize("n_steps", [384, 385, 386, 512, 513, 514, 700])
def test_step_edges(n_steps):
    wl = workloads.config2(n_particles=3, n_steps=n_steps, grid=(90, 4, 3))
    _check(wl, wl.axes)


def test_uneven_tracks():
    """Tracks shorter than a wave beside one of several blocks' runs."""
    wl = workloads.config2(n_particles=5, n_steps=2200, grid=(54, 3, 3))
    tracks = [[c[:n] for c in t[:6]] + [t[6], 0] for t, n in zip(wl.track_list(), (2200, 1, 2, 70, 900))]
    _check(wl, wl.axes, tracks=tracks)


@pytest.mark.parametrize("waves,groups", [(1, 1), (2, 5), (4, 0), (4, 24)])
def test_blocks_and_direction_groups(waves, groups):
    wl = workloads.config2(n_particles=2, n_steps=400, grid=(96, 6, 4))
    _check(wl, wl.axes, tuning=engine.Tuning(waves_per_block=waves, slices=groups))


@pytest.mark.parametrize("lo,hi", [(0.0, 6.0), (-3.0, 3.0), (-6.0, -0.5), (4.0, 0.0)])
def test_cut_steps_and_signs(lo, hi):
    """Frequencies past the steps' thresholds, on grids of either sign and order."""
    wl = workloads.config2(n_particles=2, n_steps=1100, grid=(100, 4, 3))
    top = wl.axes["omega"][-1]
    axes = dict(wl.axes, omega=np.linspace(lo * top, hi * top, 100))
    for comp in ("total", "cartesian"):
        _check(wl, axes, comp)


@pytest.mark.parametrize("comp,n_steps,it_range", [
    ("total", 500, (0, 200)), ("total", 500, (0, 300)), ("cartesian", 1100, (0, 260))])
def test_window(comp, n_steps, it_range):
    wl = workloads.config2(n_particles=2, n_steps=n_steps, grid=(210, 3, 3))
    _check(wl, wl.axes, comp, it_range=it_range)


def test_coefficients_that_are_not_finite_stay_with_the_steps_that_keep_them():
    """An infinite dL/dS at a frequency that most steps cut leaves the others' gradients finite."""
    wl = workloads.config2(n_particles=1, n_steps=500, grid=(100, 3, 2))
    top = wl.axes["omega"][-1]
    axes = dict(wl.axes, omega=np.linspace(0.0, 8.0 * top, 100))
    grid = engine.DeviceGrid("far", axes["omega"], axes["theta"], axes["phi"])
    G = torch.ones((1, 2, 3, 100), dtype=torch.float64, device="cuda")
    G[..., 99] = float("inf")
    a, b = (_grads(wl.batch, grid, [G], "total", prec) for prec in ("float", "double"))
    for c in range(3):
        assert torch.equal(torch.isfinite(a[c]), torch.isfinite(b[c]))


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("comp", ["total", "cartesian"])
def test_positions_that_are_not_finite_stay_out(comp, bad):
    """A sample at such a position keeps no frequency (nor does the one after it), so its
    gradients are zero, as in the FP64 path, also where its wave's other steps cut groups."""
    wl = workloads.config2(n_particles=1, n_steps=1100, grid=(100, 4, 3))
    axes = dict(wl.axes, omega=np.linspace(0.0, 6.0 * wl.axes["omega"][-1], 100))
    track = [np.array(c) for c in wl.track_list()[0][:6]]
    track[0][[200, 777]] = bad
    _check(wl, axes, comp, tracks=[track + [1.0, 0]])


@pytest.mark.parametrize("order", ["up", "down", "cross"])
@pytest.mark.parametrize("comp,n_omega,n_steps,it_range", [
    ("total", 24, 400, None), ("total", 31, 500, None), ("total", 48, 390, None),
    ("cartesian", 201, 1100, (0, 120)), ("cartesian", 513, 1100, (0, 250))])
def test_long_tracks_of_few_pairs(comp, n_omega, n_steps, it_range, order):
    """Few omegas, or a window of a long track: the rotation loop in FP64, here of FP64 fields.
    What a position's gradient sums is rounded to FP32 in the coefficient, the frequency, the
    sine, the cosine, two products and a run's sum: 8 roundings of 2^-24 bound it; the
    momenta's sums over the track cancel to a twentieth of their terms.  The weights' are
    FP64."""
    wl = workloads.config2(n_particles=3, n_steps=n_steps, grid=(n_omega, 4, 3))
    top = wl.axes["omega"][-1]
    omega = {"up": np.linspace(0.1, 2.0, n_omega), "down": np.linspace(2.0, 0.1, n_omega),
             "cross": np.linspace(-2.0, 2.0, n_omega)}[order] * top
    _check(wl, dict(wl.axes, omega=omega), comp, it_range=it_range, exact_fields=True,
           bars=[5e-7] * 3 + [1e-5] * 3 + [1e-12])


def test_tables_of_several_launches():
    """More tables than fit at once: 90 electrons, 32 x 32 directions, 128 frequencies."""
    wl = workloads.config2(n_particles=90, n_steps=390, grid=(128, 32, 32))
    _check(wl, wl.axes)
