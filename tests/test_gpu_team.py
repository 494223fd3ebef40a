"""The team mode of the pressure-velocity iteration (whole-GPU checks and
visits from lists while they are long, then the remaining sweeps in one
launch) against one launch per colour phase: the cell arithmetic is the same and no order shows in the
results, so every field and sweep count is equal bit for bit.  Small list
limits make the team refuse, or stop at a sweep and launches go on from it;
small maxout ends the iteration before it converges, inside either."""
import ctypes as ct
import os

import numpy as np
import pytest

from pdac_amd import abi
from pdac_amd.cases import mixed_box, shock_tube, summit_cone_3d, summit_vent_3d
from tests.golden.make_golden import load

pytestmark = pytest.mark.gpu

CASES = {
    "mixed_2d": lambda: load("mixed_2d")[0],
    "eruption_2d_vent": lambda: load("eruption_2d_vent")[0],
    "cone_3d_ib": lambda: load("cone_3d_ib")[0],
    "shock_rk3": lambda: shock_tube(nx=61, nz=7, rungekut=3, nsolid=1),
    "box_4_classes": lambda: mixed_box(three_d=True, nx=13, ny=9, nz=11, nsolid=4, seed=3),
    "box_2d_3_classes": lambda: mixed_box(nx=33, nz=21, nsolid=3, seed=5),
    "vent_odd": lambda: summit_vent_3d(nx=37, ny=41, nz=23, nsolid=2),
    "cone_40": lambda: summit_cone_3d(nx=40, ny=44, nz=30, height=230.0, sigma=230.0, rough=5.0),
    # the other mass limiters, the other pressure model, no limiter at all
    "beta": lambda: load("mixed_2d_beta")[0],
    "variants": lambda: load("mixed_2d_variants")[0],
    "van_leer_3d": lambda: mixed_box(three_d=True, nx=12, ny=9, nz=10, nsolid=2, mass_limiter=1, maxout=60),
    "superbee_3d": lambda: mixed_box(three_d=True, nx=12, ny=9, nz=10, nsolid=1, mass_limiter=3, maxout=60),
    "beta_3d": lambda: mixed_box(three_d=True, nx=9, ny=10, nz=11, nsolid=4, mass_limiter=4, beta=0.3, maxout=60),
    "ultrabeta_2d": lambda: mixed_box(nx=27, nz=24, nsolid=3, mass_limiter=0, beta=0.3, maxout=60),
    "pmodel_1_3d": lambda: mixed_box(three_d=True, nx=12, ny=9, nz=10, nsolid=3, pmodel=1),
    "pmodel_1_one_class": lambda: mixed_box(nx=26, nz=23, nsolid=1, pmodel=1),
    "muscl_off_2d": lambda: mixed_box(nx=31, nz=22, nsolid=2, muscl=0),
    "muscl_off_3d": lambda: mixed_box(three_d=True, nx=11, ny=12, nz=9, nsolid=3, muscl=0),
    # lists of a colour up to those that k_visit's waves take at two blocks a
    # compute unit (4096 cells with three classes in 3D, 2048 with four, 16384
    # with one class in 2D) and beyond them
    "box_one_round": lambda: mixed_box(three_d=True, nx=34, ny=18, nz=18, nsolid=3),
    "box_over_a_round": lambda: mixed_box(three_d=True, nx=34, ny=18, nz=19, nsolid=3),
    "box_4_classes_long": lambda: mixed_box(three_d=True, nx=28, ny=16, nz=15, nsolid=4, seed=7),
    "box_2d_long": lambda: mixed_box(nx=202, nz=172, nsolid=1),
    "maxout_1": lambda: mixed_box(three_d=True, nx=10, ny=8, nz=9, nsolid=2, maxout=1),
    "maxout_3": lambda: mixed_box(nx=24, nz=18, nsolid=2, maxout=3),
}


def solver(case, **env):
    from pdac_amd.gpu import gpu_solver
    os.environ.update(env)
    try:
        return gpu_solver(case, device=0)
    finally:
        for k in env:
            os.environ.pop(k)


def run(case, mode, limit=None, steps=3, **env):
    env["PDAC_ITER_MODE"] = mode
    if limit:
        env["PDAC_TEAM_LIMIT"] = str(limit)
    g = solver(case, **env)
    nits = [g.step(1) for _ in range(steps)]
    nits.append(g.step_by_parts())
    out = {f.lower(): g.get(f.lower()) for f in abi.FIELDS}
    total = g.nit_total
    g.close()
    return nits, total, out


@pytest.mark.parametrize("limit", [None, 1, 6, 40])
@pytest.mark.parametrize("name", sorted(CASES))
def test_team_equals_launches(name, limit):
    print(f"[team] {name} limit {limit}", flush=True)
    case = CASES[name]()
    a = run(case, "team", limit)
    b = run(case, "launches")
    assert a[0] == b[0] and a[1] == b[1], (a[:2], b[:2])
    bad = [k for k in b[2] if not np.array_equal(a[2][k], b[2][k], equal_nan=True)]
    assert not bad, bad


# PDAC_K_YGAS_FLUX and PDAC_K_ITERATE (include/pdacgpu.h)
K_YGAS_FLUX, K_ITERATE = 8, 15


def launches(g, kernel):
    n, ms = ct.c_int64(), ct.c_double()
    assert g.lib.pdac_profile_read(g.ctx, kernel, ct.byref(n), ct.byref(ms)) == 0
    return n.value


def test_long_lists_take_few_attempts():
    """Calls whose lists stay above the team's limit to the end, on a mesh
    whose sweep grid counts as not resident: the sweeps go out in batches of
    about as many as the last call took, so that a call makes a few attempts
    at a team and not one per 16 sweeps, and the step's kernels behind the
    iteration are launched once for the attempt that ends it and at most once
    in vain."""
    print("[team] long lists", flush=True)
    g = solver(CASES["cone_40"](), PDAC_TEAM_LIMIT="1", PDAC_SWEEP_EARLY="0")
    g.step(4)
    g.lib.pdac_profile_select(g.ctx, (1 << K_YGAS_FLUX) | (1 << K_ITERATE))
    g.lib.pdac_profile_enable(g.ctx, 1)
    g.lib.pdac_profile_reset(g.ctx)
    before, steps = g.nit_total, 16
    g.step(steps)
    sweeps, teams, ygas = g.nit_total - before, launches(g, K_ITERATE), launches(g, K_YGAS_FLUX)
    g.close()
    print(f"[team] {sweeps} sweeps, {teams} teams, {ygas} launches of the species fluxes in {steps} steps", flush=True)
    assert sweeps > 40 * steps
    assert teams <= 3 * steps
    assert ygas <= 2 * steps


@pytest.mark.parametrize("name", ["cone_40", "box_2d_3_classes", "maxout_3"])
def test_no_compute_units_for_a_team(name):
    """Fewer blocks than a team needs: the election finds no XCD and gives up
    after its bounded wait, the call goes on with launches, and later calls do
    not try again."""
    print(f"[team] no XCD, {name}", flush=True)
    a = run(CASES[name](), "team", PDAC_TEAM_GRID="31")
    b = run(CASES[name](), "launches")
    assert a[0] == b[0] and a[1] == b[1], (a[:2], b[:2])
    bad = [k for k in b[2] if not np.array_equal(a[2][k], b[2][k], equal_nan=True)]
    assert not bad, bad
    g = solver(CASES[name](), PDAC_TEAM_GRID="31")
    g.lib.pdac_profile_select(g.ctx, 1 << K_ITERATE)
    g.lib.pdac_profile_enable(g.ctx, 1)
    g.lib.pdac_profile_reset(g.ctx)
    g.step(8)
    teams = launches(g, K_ITERATE)
    g.close()
    # (a launch that finds its lists too long for a team holds no election)
    assert teams <= 3, teams


@pytest.mark.parametrize("value", ["0", "257", "x"])
def test_team_grid_out_of_range_is_refused(value):
    from pdac_amd.solver import PdacError
    with pytest.raises(PdacError, match="PDAC_TEAM_GRID"):
        solver(CASES["maxout_1"](), PDAC_TEAM_GRID=value)


def test_two_contexts_in_two_threads():
    """Two domains stepped at the same time from two threads, each on its own
    stream: their teams run side by side (or one does without), and each gives
    what it gives alone."""
    from concurrent.futures import ThreadPoolExecutor
    print("[team] two threads", flush=True)
    names, steps = ("cone_40", "vent_odd"), 12
    alone = {}
    for name in names:
        g = solver(CASES[name]())
        g.step(steps)
        alone[name] = (g.nit_total, g.state())
        g.close()
    pair = [solver(CASES[name]()) for name in names]
    with ThreadPoolExecutor(2) as pool:
        list(pool.map(lambda g: g.step(steps), pair))
    for name, g in zip(names, pair):
        nit, st = g.nit_total, g.state()
        g.close()
        assert nit == alone[name][0]
        for k, v in alone[name][1].items():
            np.testing.assert_array_equal(st[k], v, err_msg=k)
