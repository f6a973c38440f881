"""A second geometry on the same context: a step after it equals a step of a fresh context, and fields read before any
geometry or state are zero."""
import ctypes as C

import numpy as np
import pytest

from mflbm import Case, Simulation, geometry, native
from mflbm.native import dptr, i8ptr, iptr

pytestmark = pytest.mark.gpu


def _case(seed, porosity):
    n = (24, 20, 28)
    ctl = {"lattice_dimensions": n, "periodic_indicator": (0, 0, 1), "domain_wall_status_z": (0, 0),
           "MPI_async_layers_num": (0, 0, 4), "fluid1_viscosity": 0.1, "fluid2_viscosity": 0.08, "surface_tension": 0.02,
           "theta": 60.0, "body_force_0": 1e-5, "initial_fluid_distribution_option": 1, "initial_interface_position": 9.0}
    return Case(ctl, geometry.sphere_pack(*n, porosity, 2.0, 4.0, seed, buffer=2))


def test_second_geometry_equals_a_fresh_context():
    first, second = _case(1, 0.3), _case(2, 0.6)
    again, fresh = Simulation(first), Simulation(second)
    again.run(1, 7)
    b = second.lists
    again._call("upload_geometry", i8ptr(second.walls_h2), len(b.s_nfl), iptr(b.s_ijk), iptr(b.s_nfl), iptr(b.s_nbr),
                dptr(b.s_w), len(b.f_theta), iptr(b.f_ijk), dptr(b.f_nw), dptr(b.f_theta), dptr(second.w_in))
    again.upload(second.initial_state())
    again.color_gradient()
    for s in (again, fresh):
        s.run(1, 9)
    x, y = again.state(), fresh.state()
    fluid = second.walls_global == 0
    for key, h in (("f", 1), ("g", 1), ("phi", 4)):
        p, q = (getattr(v, key)[..., h:-h, h:-h, h:-h][..., fluid] for v in (x, y))
        assert np.array_equal(p, q), key
    again.close()
    fresh.close()


def test_fields_before_a_geometry_are_zero():
    case = _case(1, 0.3)
    lib = native.load()
    fn = native.bind(lib, "mflbm_")
    ctx = C.c_void_p()
    assert fn["create"](C.byref(case.params), C.byref(ctx)) == 0
    nz, ny, nx = case.walls_global.shape
    phi = np.full((nz + 8, ny + 8, nx + 8), 3.0)
    assert fn["download_macro"](ctx, None, None, None, None, dptr(phi)) == 0
    assert not phi.any()
    fn["destroy"](ctx)
