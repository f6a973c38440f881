"""The periodic phi halo is copied one thread a halo node inside the chain's first launch (the plan's, or with
MFLBM_CHAIN=all the whole-list one): y, z and both directions periodic, and y periodic between an open inlet and outlet,
odd sizes with partial work-groups, an interface near the periodic faces: phi, its halo and every population bit for bit
against the oracle."""
import numpy as np
import pytest

from mflbm import Case, Simulation
from oracle_backend import OracleSimulation, set_threads

pytestmark = pytest.mark.gpu


def _case(jper, kper):
    nx, ny, nz = n = (19, 13, 22)
    walls = np.zeros((nz, ny, nx), np.int8)
    walls[:, :, 0], walls[:, :, -1] = 1, 1
    walls[5:9, 3:7, 6:12] = 1
    if not jper:
        walls[:, 0], walls[:, -1] = 1, 1
    ctl = {"lattice_dimensions": n, "periodic_indicator": (0, jper, kper), "domain_wall_status_z": (0, 0),
           "domain_wall_status_y": (0, 0) if jper else (1, 1),
           "MPI_async_layers_num": (0, 0, 0), "fluid1_viscosity": 0.1, "fluid2_viscosity": 0.08, "surface_tension": 0.02,
           "theta": 60.0, "initial_fluid_distribution_option": 1, "initial_interface_position": 5.0}
    if kper:
        ctl["body_force_0"] = 1e-5
    else:
        ctl.update(inlet_BC=1, outlet_BC=1, capillary_number=5e-3, saturation_injection=1.0, excluded_layers=(2, 2))
    return Case(ctl, walls)


@pytest.mark.parametrize("chain", [None, "all"])
@pytest.mark.parametrize("jper,kper", [(1, 0), (0, 1), (1, 1)])
def test_periodic_halo_is_bit_identical_to_the_oracle(jper, kper, chain, monkeypatch):
    print(f"[wrap halo] y {jper} z {kper} chain {chain}", flush=True)
    if chain:
        monkeypatch.setenv("MFLBM_CHAIN", chain)
    set_threads(16)
    gpu, ora = Simulation(_case(jper, kper)), OracleSimulation(_case(jper, kper))
    for t in range(1, 26):
        gpu.step(t)
        ora.step(t)
    a, b = gpu.state(), ora.state()
    for key in ("f", "g", "phi"):
        assert np.array_equal(getattr(a, key).view(np.uint64), getattr(b, key).view(np.uint64)), key
    gpu.close()
    ora.close()
