"""Device memory of a two-phase run: what is kept per lattice node (populations and phi as uploaded, the normals and
fields, walls, index tables) and per fluid node.  A lattice that is nearly all solid takes little beyond the former, so
the largest lattice that fits a device does not depend on arrays sized for a fluid node everywhere."""
import numpy as np
import pytest

from mflbm import Case, Simulation

pytestmark = pytest.mark.gpu


def test_a_solid_lattice_takes_the_dense_arrays_alone():
    import torch
    n = 300
    walls = np.ones((n, n, n), np.int8)
    walls[:, 140:160, 140:160] = 0
    ctl = {"lattice_dimensions": (n, n, n), "periodic_indicator": (0, 0, 1), "domain_wall_status_z": (0, 0),
           "MPI_async_layers_num": (0, 0, 4), "initial_fluid_distribution_option": 1, "initial_interface_position": 20.0}
    case = Case(ctl, walls, geometry="device")
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    sim = Simulation(case, device_init=True)
    sim.synchronize()
    used = before - torch.cuda.mem_get_info()[0]
    sim.run(1, 2)
    sim.close()
    total = ((n + 35) // 16 * 16) * (n + 8) ** 2
    per = used / total
    print(f"[device memory] {used / 1e9:.3f} GB, {per:.2f} bytes a padded node", flush=True)
    # 38 + 11 doubles, walls 1, index tables 4 + 0.5 + 4, brick tables 0.7, 120000 fluid nodes at most 600 bytes each, and
    # the allocator's granularity
    assert per < 402.2 + (120000 * 600 + (32 << 20)) / total
