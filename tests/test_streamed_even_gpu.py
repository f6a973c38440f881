"""Even steps of states beyond 160 MiB read and write their slots past the caches: the same values as the cached steps.

A lattice whose walls and state repeat along the periodic z direction holds copies of a small lattice's solution, which
the cached kernels compute: its copies bit for bit, in every precision, for the two-phase and single-phase programs and
the batch, and for a batch that changes from streamed to cached steps when its largest sample has converged."""
import numpy as np
import pytest

from mflbm import Case, Simulation, geometry
from mflbm.batch import REVBatch, REVSample
from mflbm.case import State
from mflbm.singlephase import SPCase, SPSimulation

pytestmark = pytest.mark.gpu

LIMIT = 160 << 20
W = np.array([1 / 3] + [1 / 18] * 6 + [1 / 36] * 12)
PRECISIONS = ["fp64", "fp32", "mixed"]


def _copies_equal(big, small, fluid, nz, halo):
    """The interior fluid nodes of every copy in ``big`` (..., z, y, x with this halo) equal ``small``'s."""
    a = small[..., halo:-halo, halo:-halo, halo:-halo]
    for k in range((big.shape[-3] - 2 * halo) // nz):
        b = big[..., halo + k * nz:halo + (k + 1) * nz, halo:-halo, halo:-halo]
        assert np.array_equal(a[..., fluid], b[..., fluid]), f"copy {k}"


def _single(walls, precision):
    nz, ny, nx = walls.shape
    ctl = {"lattice_dimensions": (nx, ny, nz), "periodic_indicator": (0, 0, 1), "domain_wall_status_z": (0, 0),
           "MPI_async_layers_num": (0, 0, 4), "fluid_viscosity": 0.1, "body_force_0": 1e-4}
    return SPCase(ctl, walls, precision)


@pytest.mark.parametrize("steps", [6, 7])
@pytest.mark.parametrize("precision", PRECISIONS)
def test_single_phase_copies(precision, steps):
    nz, k = 20, 10 if precision == "fp64" else 20
    walls = geometry.sphere_pack(128, 96, nz, 0.4, 3.0, 6.0, 3, buffer=2)
    small, big = _single(walls, precision), _single(np.tile(walls, (k, 1, 1)), precision)
    fluid = small.walls_global == 0
    size = 19 * (8 if precision == "fp64" else 4) * int(fluid.sum())
    assert size < LIMIT < k * size
    print(f"[streamed] single phase {precision} {k * size / 2**20:.0f} MiB", flush=True)
    f = []
    for c in (big, small):
        s = SPSimulation(c)
        s.run(1, steps)
        f.append(s.state().f)
        s.close()
    _copies_equal(*f, fluid, nz, 1)


@pytest.mark.parametrize("precision", PRECISIONS)
def test_batch_copies(precision):
    nz, k = 20, 10 if precision == "fp64" else 20
    walls = geometry.sphere_pack(128, 96, nz, 0.4, 3.0, 6.0, 4, buffer=2)
    fluid = _single(walls, precision).walls_global == 0
    assert 19 * (8 if precision == "fp64" else 4) * int(fluid.sum()) * k > LIMIT
    print(f"[streamed] batch {precision}", flush=True)
    both = REVBatch([REVSample(walls), REVSample(np.tile(walls, (k, 1, 1)))], 0.1, 1e-4, precision)
    alone = REVBatch([REVSample(walls)], 0.1, 1e-4, precision)
    for b in (both, alone):
        b.run(1, 8)
    want = alone.state(0)
    _copies_equal(both.state(0), want, fluid, nz, 1)
    _copies_equal(both.state(1), want, fluid, nz, 1)
    both.close()
    alone.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_batch_continues_with_cached_steps_when_its_large_sample_is_done(precision):
    """Narrow channels (large, done first) beside a duct (small, done later): the duct stops where it stops alone."""
    nz = 24
    duct = np.zeros((nz, 24, 24), np.int8)
    nzb = 76 if precision == "fp64" else 152
    narrow = np.zeros((nzb, 128, 145), np.int8)
    narrow[:, :, ::6] = 1
    fluid = _single(duct, precision).walls_global == 0
    nf = int((_single(narrow, precision).walls_global == 0).sum())
    assert 19 * (8 if precision == "fp64" else 4) * nf > LIMIT
    print(f"[streamed] batch {precision} to its end", flush=True)
    both = REVBatch([REVSample(narrow), REVSample(duct)], 0.1, 1e-5, precision, ntime_monitor=100, tol=1e-5, rest_state=1)
    alone = REVBatch([REVSample(duct)], 0.1, 1e-5, precision, ntime_monitor=100, tol=1e-5, rest_state=1)
    r, ra = both.run_steady(20000), alone.run_steady(20000)
    print(r.conv_step, ra.conv_step, flush=True)
    assert 0 < r.conv_step[0] < r.conv_step[1] == ra.conv_step[0]
    assert r.flowrate[1] == ra.flowrate[0]
    _copies_equal(both.state(1), alone.state(0), fluid, nz, 1)
    # again from the first samples' states: every sample runs, the batch streams again
    both.reset_monitor()
    r2 = both.run_steady(200)
    assert r2.periods == 2
    both.close()
    alone.close()


@pytest.mark.parametrize("steps", [2, 3])
@pytest.mark.parametrize("precision", PRECISIONS)
def test_two_phase_copies(precision, steps):
    """Walls uniform along z (a random pattern of columns), phi random at every node of the period.  An upload rounds the
    exchanged halo populations to FP32 storage apart from their images, so the copies next to the periodic faces may
    differ there in the last bit: the inner ones, 24 layers from either face, are compared (a step carries a
    difference over fewer than 8)."""
    nx, ny, nz = 112, 96, 24
    few, many = (3, 6) if precision == "fp64" else (4, 9)
    rng = np.random.default_rng(8)
    walls = np.repeat((rng.random((1, ny, nx)) < 0.35).astype(np.int8), nz, 0)
    phi = rng.uniform(-1.0, 1.0, (nz, ny, nx))
    out = []
    for m in (many, few):
        ctl = {"lattice_dimensions": (nx, ny, m * nz), "periodic_indicator": (0, 0, 1), "domain_wall_status_z": (0, 0),
               "MPI_async_layers_num": (0, 0, 4), "fluid1_viscosity": 0.1, "fluid2_viscosity": 0.08, "surface_tension": 0.02,
               "theta": 60.0, "body_force_0": 1e-5, "initial_fluid_distribution_option": 1, "initial_interface_position": 8.0}
        case = Case(ctl, np.tile(walls, (m, 1, 1)), precision=precision)
        fluid = case.walls_global[:nz] == 0
        st = State.empty(nx, ny, m * nz)
        at = np.arange(-4, m * nz + 4) % nz
        st.phi[:, 4:-4, 4:-4] = np.where(fluid, phi, 0.0)[at]
        for q in range(19):
            st.f[q] = W[q] * 0.5 * (1.0 + st.phi[3:-3, 3:-3, 3:-3])
            st.g[q] = W[q] * 0.5 * (1.0 - st.phi[3:-3, 3:-3, 3:-3])
        size = 19 * (16 if precision == "fp64" else 8) * int(fluid.sum())
        assert few * size < LIMIT < many * size
        print(f"[streamed] two phase {precision} {m * size / 2**20:.0f} MiB", flush=True)
        s = Simulation(case, state=st)
        s.run(1, steps)
        out.append(s.state())
        s.close()
    for key, halo in (("f", 1), ("g", 1), ("phi", 4)):
        a, b = getattr(out[0], key), getattr(out[1], key)
        assert np.isfinite(b).all()
        inner = lambda v, k, n: v[..., k * nz:(k + n) * nz + 2 * halo, :, :]
        _copies_equal(inner(a, 1, many - 2), inner(b, 1, 1), fluid, nz, halo)


def test_late_steps_of_a_batch_cost_what_the_running_sample_costs():
    """A duct of 154 MB (FP32, cached by itself) beside narrow channels of 217 MB that converge first: from then on a
    step takes as long as in a batch of the duct alone (streaming a state that the cache holds costs 12 %)."""
    import time
    narrow = np.zeros((152, 152, 152), np.int8)
    narrow[:, :, ::6] = 1
    duct = np.zeros((128, 128, 128), np.int8)
    us = []
    for samples in ([REVSample(narrow), REVSample(duct)], [REVSample(duct)]):
        b = REVBatch(samples, 0.1, 1e-6, "fp32", ntime_monitor=200, tol=1e-4, rest_state=1)
        r = b.run_steady(1600)
        assert all(r.conv_step[:-1] > 0) and r.conv_step[-1] == 0
        ts = []
        for _ in range(6):
            t = time.perf_counter()
            b.run_steady(2000)
            ts.append((time.perf_counter() - t) / 2000 * 1e6)
        us.append(min(ts))
        assert b.results().conv_step[-1] == 0
        b.close()
    print(f"[streamed] late steps {us[0]:.1f} us, alone {us[1]:.1f} us", flush=True)
    assert us[0] < 1.1 * us[1]
