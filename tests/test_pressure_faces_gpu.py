"""The pressure (Zou-He) inlet and outlet hold the 19 slots of a face node in registers.  Boxes with solid and fluid face
nodes, faces of less and more than one work-group, a pressure outlet with a pressure and with a velocity inlet: every
population and phi bit for bit against the oracle, after an even and after an odd last step."""
import numpy as np
import pytest

from mflbm import Case, Simulation, geometry
from oracle_backend import OracleSimulation, set_threads

pytestmark = pytest.mark.gpu


def _case(n, inlet, outlet):
    walls = geometry.sphere_pack(*n, 0.35, 2.0, 4.0, 9, buffer=0)
    ctl = {"lattice_dimensions": n, "periodic_indicator": (0, 0, 0), "domain_wall_status_z": (0, 0),
           "MPI_async_layers_num": (0, 0, 0), "inlet_BC": inlet, "outlet_BC": outlet, "fluid1_viscosity": 0.1,
           "fluid2_viscosity": 0.08, "surface_tension": 0.02, "theta": 60.0, "capillary_number": 5e-3,
           "initial_fluid_distribution_option": 1, "initial_interface_position": 5.0, "saturation_injection": 1.0,
           "excluded_layers": (2, 2)}
    return Case(ctl, walls)


@pytest.mark.parametrize("inlet,outlet", [(2, 2), (1, 2)])
@pytest.mark.parametrize("n,nsteps", [((13, 15, 24), 30), ((35, 20, 18), 31)])
def test_pressure_faces_are_bit_identical_to_the_oracle(n, nsteps, inlet, outlet):
    print(f"[pressure faces] {n} inlet {inlet} outlet {outlet}", flush=True)
    set_threads(16)
    gpu, ora = Simulation(_case(n, inlet, outlet)), OracleSimulation(_case(n, inlet, outlet))
    for t in range(1, nsteps + 1):
        gpu.step(t)
        ora.step(t)
    a, b = gpu.state(), ora.state()
    for key in ("f", "g", "phi"):
        assert np.array_equal(getattr(a, key).view(np.uint64), getattr(b, key).view(np.uint64)), key
    gpu.close()
    ora.close()
