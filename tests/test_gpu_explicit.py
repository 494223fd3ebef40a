"""Parity of the explicit Runge-Kutta step (explicit_solver.f,
time_integration = 1) of the HIP library with the CPU checker and with the
reference solver's golden fixtures.

The GPU runs the reference's stage order (every cell's gas-enthalpy pressure
work reads its west/south/bottom neighbours as already updated in the same
stage), so it follows the reference operation for operation.  The bound is
the explicit-step bar, 1e-12 relative per field: the only differences come
from pow/exp/sqrt of the device and host math libraries (viscon, Gunn's
correlation, the drag laws), which differ in the last bits.

* subroutine by subroutine within each step, from a common state at the
  start of the step (the Runge-Kutta star state lives inside each library,
  so states are re-synchronised only between steps);
* whole steps against the reference's fixtures and against the checker;
* the stage-start order (PDAC_ORDER_STAGE) against the checker in that order;
* the chain of the reference order by its three kernels (fixed-point
  iterates, serial anti-diagonals, generic);
* a 48x96 eruption column over 20 steps against the checker;
* the FP32-flux form against the FP64 form.
"""
import numpy as np
import pytest

from oracle.binding import cpu_solver
from pdac_amd import abi
from tests.golden.make_golden import CASES, load

pytestmark = pytest.mark.gpu

EXPLICIT = sorted(n for n in CASES if n.startswith("explicit_"))
TOL = 1e-12


def gpu(case, **kw):
    from pdac_amd.gpu import gpu_solver
    return gpu_solver(case, device=0, **kw)


def rel(a, b):
    a = np.asarray(a, dtype=np.float64)
    b = np.asarray(b, dtype=np.float64)
    scale = np.max(np.abs(b)) if b.size else 0.0
    d = np.max(np.abs(a - b)) if b.size else 0.0
    return d / scale if scale > 0.0 else d


def all_fields(s):
    return {name.lower(): s.get(name.lower()) for name in abi.FIELDS}


def sync(g, c):
    for name in abi.FIELDS:
        g.put(name.lower(), c.get(name.lower()))


def compare(g, c, tol, where, skip=()):
    fg, fc = all_fields(g), all_fields(c)
    bad = {k: rel(fg[k], fc[k]) for k in fc if k not in skip and rel(fg[k], fc[k]) > tol}
    assert not bad, f"{where}: " + ", ".join(f"{k}={v:.2e}" for k, v in sorted(bad.items()))


# fields the explicit step does not maintain (semi-implicit work arrays)
SEMI_ONLY = ("rugn", "rvgn", "rwgn", "rusn", "rvsn", "rwsn", "rug", "rvg", "rwg", "rus", "rvs",
             "rws", "rhg", "rhs")


@pytest.mark.parametrize("name", EXPLICIT)
def test_subroutines(name):
    print(f"[explicit subroutines] {name}", flush=True)
    case, _, _ = load(name)
    g, c = gpu(case), cpu_solver(case, iter_order=abi.ORDER_LEXICOGRAPHIC)
    sync(g, c)
    dt = case.dt
    rk_n = case.rungekut
    for step in range(case.nsteps):
        for s in (g, c):
            s.boundary()
        compare(g, c, TOL, f"{name} step {step} boundary", SEMI_ONLY)
        for s in (g, c):
            s.initialize_fieldn(dt)
        compare(g, c, TOL, f"{name} step {step} initialize_fieldn", SEMI_ONLY)
        for rk in range(1, rk_n + 1):
            dts = dt / (rk_n + 1 - rk)
            fg, cg = g.explicit_iter(dts)
            fc, cc = c.explicit_iter(dts)
            assert fg == fc, (fg, fc)
            assert abs(cg - cc) <= TOL * abs(cc), (cg, cc)
            assert cc > 0.0
            compare(g, c, TOL, f"{name} step {step} explicit_iter {rk}", SEMI_ONLY)
            for s in (g, c):
                s.ygas(dts)
            compare(g, c, TOL, f"{name} step {step} ygas {rk}", SEMI_ONLY)
        sync(g, c)
    g.close()
    c.close()


@pytest.mark.parametrize("name", EXPLICIT)
def test_steps_match_reference(name):
    print(f"[explicit reference] {name}", flush=True)
    case, ref, _ = load(name)
    g = gpu(case)
    g.step(case.nsteps)
    out = g.state()
    g.close()
    for k, v in ref.items():
        assert rel(out[k].reshape(v.shape), v) <= TOL, (k, rel(out[k].reshape(v.shape), v))


@pytest.mark.parametrize("name", EXPLICIT)
def test_stage_order_matches_checker(name):
    print(f"[explicit stage order] {name}", flush=True)
    case, ref, _ = load(name)
    g = gpu(case, iter_order=abi.ORDER_STAGE)
    c = cpu_solver(case, iter_order=abi.ORDER_STAGE)
    g.step(case.nsteps)
    c.step(case.nsteps)
    sg, sc = g.state(), c.state()
    g.close()
    c.close()
    for k in sc:
        assert rel(sg[k], sc[k]) <= TOL, (k, rel(sg[k], sc[k]))
    # and it is a different order from the reference's
    assert max(rel(sg[k].reshape(v.shape), v) for k, v in ref.items()) > 1e-10


@pytest.mark.parametrize("mode", ["serial", "1"])
@pytest.mark.parametrize("name", EXPLICIT)
def test_chain_kernels_match_reference(name, mode, monkeypatch):
    """The default evaluates the reference order's chain as a fixed point of
    all-cells iterates; the serial chain (PDAC_CHAIN=serial, the last resort of
    the fixed point) and one iterate with the rest done by one work-group
    (PDAC_CHAIN=1) must give the fixtures' fields as well."""
    print(f"[explicit chain {mode}] {name}", flush=True)
    monkeypatch.setenv("PDAC_CHAIN", mode)
    case, ref, _ = load(name)
    g = gpu(case)
    g.step(case.nsteps)
    out = g.state()
    g.close()
    for k, v in ref.items():
        assert rel(out[k].reshape(v.shape), v) <= TOL, (k, rel(out[k].reshape(v.shape), v))


def test_chain_fixed_point_equals_serial(monkeypatch):
    """Fixed-point iterates and the serial chain agree bit for bit on a 48x96
    eruption column over 10 steps."""
    from pdac_amd.cases import eruption_column
    print("[explicit chain fixed point vs serial]", flush=True)
    out = {}
    for mode in ("serial", "fixed"):
        if mode == "serial":
            monkeypatch.setenv("PDAC_CHAIN", "serial")
        else:
            monkeypatch.delenv("PDAC_CHAIN", raising=False)
        case = eruption_column(nx=48, nz=96, nsteps=10, dt=5.0e-5, vent_radius=10.0)
        case.time_integration = 1
        g = gpu(case)
        g.step(case.nsteps)
        out[mode] = g.state()
        g.close()
    for k in out["serial"]:
        np.testing.assert_array_equal(out["fixed"][k], out["serial"][k], err_msg=k)


def test_eruption_column_20_steps():
    from pdac_amd.cases import eruption_column
    print("[explicit eruption 48x96]", flush=True)
    case = eruption_column(nx=48, nz=96, nsteps=20, dt=5.0e-5, vent_radius=10.0)
    case.time_integration = 1
    g, c = gpu(case), cpu_solver(case, iter_order=abi.ORDER_LEXICOGRAPHIC)
    g.step(case.nsteps)
    c.step(case.nsteps)
    sg, sc = g.state(), c.state()
    g.close()
    c.close()
    init = case.fields
    assert max(rel(sc[k], init[k]) for k in ("p", "wg")) > 1e-6  # the column moved
    for k in sc:
        assert rel(sg[k], sc[k]) <= 1e-11, (k, rel(sg[k], sc[k]))


def rel_l2(a, b):
    a = np.asarray(a, dtype=np.float64).reshape(-1)
    b = np.asarray(b, dtype=np.float64).reshape(-1)
    nb = np.linalg.norm(b)
    return np.linalg.norm(a - b) / nb if nb > 0 else np.linalg.norm(a - b)


def test_fp32flux_form_error():
    """FP32 momentum/enthalpy flux arithmetic in the explicit step: relative
    L2 error of p and of each particle volume fraction at most 1e-4 against
    the FP64 form, every field within 1e-3."""
    from pdac_amd.cases import eruption_column
    print("[explicit fp32flux]", flush=True)
    case = eruption_column(nx=48, nz=96, nsteps=50, dt=5.0e-5, vent_radius=10.0)
    case.time_integration = 1
    out = {}
    for prec in (abi.PREC_FP32FLUX, abi.PREC_FP64):
        s = gpu(case, precision=prec)
        s.step(case.nsteps)
        out[prec] = s.state()
        s.close()
    a, b = out[abi.PREC_FP32FLUX], out[abi.PREC_FP64]
    e = {k: rel_l2(a[k], b[k]) for k in b}
    rho = np.asarray(case.density[:case.nsolid]).reshape(-1, 1)
    e["eps_s"] = max(rel_l2(a["rlk"].reshape(case.nsolid, -1)[s] / rho[s],
                            b["rlk"].reshape(case.nsolid, -1)[s] / rho[s])
                     for s in range(case.nsolid))
    print(" ".join(f"{k}:{v:.1e}" for k, v in sorted(e.items())), flush=True)
    assert e["p"] <= 1e-4 and e["eps_s"] <= 1e-4, e
    assert max(e.values()) <= 1e-3, e
    assert max(e.values()) > 0.0
