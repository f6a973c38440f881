"""The chain's plan lists runs of entries: consecutive bricks (16 x 2 x 2 nodes) of a tile's row of 8 bricks, across bricks
without entries, in pieces of 64.  Boxes whose rows of bricks end inside a tile (2, 3 and 9 bricks) and whose brick rows
and layers leave partial tiles, with an interface crossing the rows at an angle, so that runs begin and end inside them:
every population, phi and normal bit for bit against the oracle, which evaluates every node."""
import numpy as np
import pytest

from mflbm import Case, Simulation, geometry
from oracle_backend import OracleSimulation, set_threads

pytestmark = pytest.mark.gpu


def _case(n, packed):
    nx, ny, nz = n
    if packed:
        walls = geometry.sphere_pack(nx, ny, nz, 0.4, 2.0, 5.0, 5, buffer=4)
    else:   # an open channel: most bricks hold no solid entries
        walls = np.zeros((nz, ny, nx), np.int8)
        walls[:, :, 0], walls[:, :, -1] = 1, 1
        walls[:, 0], walls[:, -1] = 1, 1
    ctl = {"lattice_dimensions": n, "periodic_indicator": (0, 0, 0), "domain_wall_status_z": (0, 0),
           "MPI_async_layers_num": (0, 0, 0), "inlet_BC": 1, "outlet_BC": 1, "fluid1_viscosity": 0.1,
           "fluid2_viscosity": 0.1, "surface_tension": 0.02, "theta": 40.0, "capillary_number": 5e-3,
           "initial_fluid_distribution_option": 1, "initial_interface_position": 5.0, "saturation_injection": 1.0,
           "excluded_layers": (4, 4)}
    return Case(ctl, walls)


@pytest.mark.parametrize("n,packed", [((18, 19, 40), True), ((140, 21, 30), True), ((140, 21, 30), False), ((35, 40, 33), False)])
def test_runs_of_bricks_are_bit_identical_to_the_oracle(n, packed):
    print(f"[chain runs] {n} packed {packed}", flush=True)
    set_threads(16)
    gpu, ora = Simulation(_case(n, packed)), OracleSimulation(_case(n, packed))
    for t in range(1, 61):
        gpu.step(t)
        ora.step(t)
    a, b = gpu.state(), ora.state()
    for key in ("f", "g", "phi"):
        assert np.array_equal(getattr(a, key).view(np.uint64), getattr(b, key).view(np.uint64)), key
    ga, gb = gpu.gradient(), ora.gradient()
    for k in ga:
        assert np.array_equal(ga[k], gb[k]), k
    gpu.close()
    ora.close()
