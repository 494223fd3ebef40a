"""The explicit step's chain as a fixed point (2D, 3D, ensembles and
pdac_explicit_step_noalloc): equal bit for bit to the serial chain kernel
(PDAC_CHAIN=general), whose order the reference's is, also where the iterates
launched do not reach it and one work-group goes on (PDAC_CHAIN=1, 2)."""
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


def chain(monkeypatch, mode):
    if mode is None:
        monkeypatch.delenv("PDAC_CHAIN", raising=False)
    else:
        monkeypatch.setenv("PDAC_CHAIN", mode)


def run(case, monkeypatch, general, noalloc=False, steps=4):
    from pdac_amd.gpu import gpu_solver, lib
    chain(monkeypatch, {True: "general", False: None}.get(general, general))
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


@pytest.mark.parametrize("iterates", ["1", "2"])
@pytest.mark.parametrize("name", ["box_3d_3_classes", "wide_2d", "column_2d"])
def test_one_work_group_goes_on(name, iterates, monkeypatch):
    print(f"[chain fixed point] {name} after {iterates}", flush=True)
    def case():
        if name != "column_2d":
            return CASES[name]()
        c = eruption_column(nx=24, nz=40, dt=2.0e-4, vent_radius=6.0)
        c.time_integration = 1
        return c
    a = run(case(), monkeypatch, iterates)
    b = run(case(), monkeypatch, "general")
    for k in b:
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)


@pytest.mark.parametrize("mode", [None, "1"])
def test_ensemble_of_3d_members(mode, monkeypatch):
    from pdac_amd.gpu import Ensemble, gpu_solver
    print(f"[chain fixed point] 3D ensemble {mode}", flush=True)
    mk = lambda: [vent(), vent(), box(three_d=True, nx=9, ny=12, nz=5, nsolid=2)]
    want = [run(c, monkeypatch, True, steps=3) for c in mk()]
    chain(monkeypatch, mode)
    ms = [gpu_solver(c, device=0) for c in mk()]
    e = Ensemble(ms)
    e.step(3)
    for m, w in zip(ms, want):
        got = m.state()
        for k in got:
            np.testing.assert_array_equal(got[k], w[k], err_msg=k)
        m.close()
    e.close()


def test_pressures_that_are_not_numbers(monkeypatch):
    """A state whose pressures have become NaN (its steps report the failure of
    the equation of state): the iterates compare bits, so a NaN that stays is
    no change, the stages are done after a few iterates again and the fields
    are the serial chain's."""
    from pdac_amd.gpu import gpu_solver
    from pdac_amd.solver import PdacError
    print("[chain fixed point] NaN pressures", flush=True)
    K_XCHAIN = 19  # PDAC_K_XCHAIN, include/pdacgpu.h
    out, launches = {}, {}
    for mode in (None, "general"):
        chain(monkeypatch, mode)
        c = eruption_column(nx=24, nz=40, dt=2.0e-4, vent_radius=6.0)
        c.time_integration = 1
        g = gpu_solver(c, device=0)
        p = g.get("p")
        p.reshape(-1)[3 * c.nx + 3] = np.nan
        g.put("p", p)
        for step in range(12):
            if step == 10:
                g.lib.pdac_profile_select(g.ctx, 1 << K_XCHAIN)
                g.lib.pdac_profile_enable(g.ctx, 1)
                g.lib.pdac_profile_reset(g.ctx)
            try:
                g.step(1)
            except PdacError as e:
                assert "equation of state" in str(e)
        n, ms = ct.c_int64(), ct.c_double()
        assert g.lib.pdac_profile_read(g.ctx, K_XCHAIN, ct.byref(n), ct.byref(ms)) == 0
        launches[mode] = n.value
        out[mode] = {k: g.get(k) for k in ("p", "tg", "sieg", "cg", "ug", "rlk")}
        g.close()
    print(f"[chain fixed point] chain launches of two steps: {launches}", flush=True)
    assert np.isnan(out[None]["p"]).any()
    for k, v in out["general"].items():
        np.testing.assert_array_equal(out[None][k], v, err_msg=k)
    # two chained stages a step: a few iterates and two more launches in each
    assert launches[None] <= 2 * 2 * 20
