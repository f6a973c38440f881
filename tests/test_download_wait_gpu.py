"""A download behind queued steps waits for them on one thread: the copying threads start when the first piece of a field
has arrived, so the wait costs the host at most the waiting thread and the runtime's own."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_waiting_for_queued_steps_keeps_few_threads_busy():
    from mflbm.singlephase import SPCase, SPSimulation
    n = (128, 128, 160)
    ctl = {"lattice_dimensions": n, "periodic_indicator": (0, 0, 1), "domain_wall_status_z": (0, 0),
           "MPI_async_layers_num": (0, 0, 4), "fluid_viscosity": 0.1, "body_force_0": 1e-6}
    sim = SPSimulation(SPCase(ctl, np.zeros(n[::-1], np.int8)))
    sim.state()   # the ring, and the pages of the first arrays
    sim.run(1, 2)
    sim.synchronize()
    t, c = time.perf_counter(), time.process_time()
    sim.run(3, 20000)
    sim.state()
    wall, cpu = time.perf_counter() - t, time.process_time() - c
    sim.close()
    print(f"[download wait] {wall:.2f} s, {cpu:.2f} s of processor time", flush=True)
    assert wall > 0.7      # (the steps were queued, not done, when the download began)
    assert cpu < 3.0 * wall
