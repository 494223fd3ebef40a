"""The team kernel of the pressure-velocity iteration (the sweeps after the
first ones in one launch, from lists of the flagged cells) against one launch
per colour phase: the cell arithmetic is the same and no order shows in the
results, so every field and sweep count is equal bit for bit.  Small list
limits make the team refuse, or stop at a sweep and launches go on from it;
small maxout ends the iteration before it converges, inside either."""
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
    "maxout_1": lambda: mixed_box(three_d=True, nx=10, ny=8, nz=9, nsolid=2, maxout=1),
    "maxout_3": lambda: mixed_box(nx=24, nz=18, nsolid=2, maxout=3),
}


def run(case, mode, limit=None, steps=3):
    from pdac_amd.gpu import gpu_solver
    env = {"PDAC_ITER_MODE": mode}
    if limit:
        env["PDAC_TEAM_LIMIT"] = str(limit)
    os.environ.update(env)
    try:
        g = gpu_solver(case, device=0)
    finally:
        for k in env:
            os.environ.pop(k)
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
