"""The explicit step's chain as a fixed point on the meshes that the 2D
diagonal-major kernels do not take (3D, more than 512 columns, and
pdac_explicit_step_noalloc): equal bit for bit to the serial chain kernel
(PDAC_CHAIN=general), whose order the reference's is."""
import ctypes as ct

import numpy as np
import pytest

from pdac_amd.cases import eruption_column, mixed_box, summit_vent_3d

pytestmark = pytest.mark.gpu


def box(**kw):
    case = mixed_box(**kw)
    case.time_integration = 1
    return case


def vent():
    case = summit_vent_3d(nx=19, ny=23, nz=17, nsolid=2, vent_half=30.0)
    case.time_integration = 1
    case.dt = 1.0e-3
    return case


def wide():
    case = eruption_column(nx=531, nz=13, dr0=2.0, dr1=2.0, dt=1.0e-4, vent="inlet")
    case.time_integration = 1
    return case


CASES = {
    "smallest_3d": lambda: box(three_d=True, nx=4, ny=4, nz=4, nsolid=1),
    "box_3d_3_classes": lambda: box(three_d=True, nx=11, ny=6, nz=21, nsolid=3),
    "box_3d_muscl_off": lambda: box(three_d=True, nx=9, ny=12, nz=5, nsolid=2, muscl=0, rungekut=2),
    "vent_3d_inlets": vent,
    "wide_2d": wide,
}


def run(case, monkeypatch, general, noalloc=False, steps=4):
    from pdac_amd.gpu import gpu_solver, lib
    if general:
        monkeypatch.setenv("PDAC_CHAIN", "general")
    else:
        monkeypatch.delenv("PDAC_CHAIN", raising=False)
    g = gpu_solver(case, device=0)
    if noalloc:
        fail, cfl = ct.c_int32(), ct.c_double()
        assert lib().pdac_explicit_step_noalloc(g.ctx, case.dt, case.rungekut, steps, ct.byref(fail), ct.byref(cfl)) == 0
    else:
        for _ in range(steps):
            g.step(1)
    out = g.state()
    out["cg"] = g.get("cg")
    g.close()
    return out


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("name", sorted(CASES))
def test_fixed_point_equals_serial_chain(name, noalloc, monkeypatch):
    print(f"[chain fixed point] {name} noalloc {noalloc}", flush=True)
    a = run(CASES[name](), monkeypatch, False, noalloc)
    b = run(CASES[name](), monkeypatch, True)
    for k in b:
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)
