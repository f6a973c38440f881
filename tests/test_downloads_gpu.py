"""State downloads through the chunked pinned ring: what was uploaded comes back bit for bit when a box is smaller than
a chunk, exactly a chunk, one element more than whole chunks and many chunks long (chunk: 2^19 elements), for the
single-phase state, and the two-phase state whose phi has another halo."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(3, 4, 12), (62, 62, 126), (61, 63, 127), (97, 83, 151)])
def test_single_phase_state_round_trip(shape):
    from mflbm.singlephase import SPCase, SPSimulation, SPState
    nx, ny, nz = shape
    ctl = {"lattice_dimensions": shape, "periodic_indicator": (0, 0, 1), "domain_wall_status_z": (0, 0),
           "MPI_async_layers_num": (0, 0, 4), "fluid_viscosity": 0.1, "body_force_0": 1e-6}
    case = SPCase(ctl, np.zeros((nz, ny, nx), np.int8))
    rng = np.random.default_rng(nx)
    st = SPState(rng.random((19, nz + 2, ny + 2, nx + 2)), np.zeros((19, ny + 2, nx + 2)))
    sim = SPSimulation(case, st)   # (before the first step of a z-periodic run the state comes back as given)
    got = sim.state().f
    sim.close()
    assert np.array_equal(got, st.f)


def test_two_phase_state_and_gradient_round_trip():
    from mflbm import Case, Simulation
    nx, ny, nz = 70, 61, 135
    ctl = {"lattice_dimensions": (nx, ny, nz), "periodic_indicator": (0, 0, 1), "domain_wall_status_z": (0, 0),
           "MPI_async_layers_num": (0, 0, 4), "initial_fluid_distribution_option": 5, "initial_interface_position": 20.0}
    case = Case(ctl, np.zeros((nz, ny, nx), np.int8))
    st = case.initial_state()
    sim = Simulation(case, state=st)
    got, gr = sim.state(), sim.gradient()
    sim.close()
    assert np.array_equal(got.f, st.f) and np.array_equal(got.g, st.g)
    inner = np.s_[4:-4, 4:-4, 4:-4]
    fluid = case.walls_global == 0
    assert np.array_equal(got.phi[inner][fluid], st.phi[inner][fluid])
    n = gr["cn_x"] ** 2 + gr["cn_y"] ** 2 + gr["cn_z"] ** 2
    near = gr["c_norm"] > 0
    assert near.any() and np.allclose(n[near], 1.0, atol=1e-12)
