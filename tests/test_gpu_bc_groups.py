"""Boundary ranges that meet: ranges are applied several to a launch, and the
result has to be that of applying them one after the other, also where they
share points, overlap or read each other's ghosts."""
import numpy as np
import pytest

import ostc
from ostc import cases
from helpers import BV_GROUPS, grouped, oracle_zone

pytestmark = pytest.mark.gpu

EXTRA = {
    # an outflow patch under the wall: the later wall overwrites it
    "overlap": [dict(type=6, raw=(5, 12, 0, 0, 0, 0), label=6)],
    # two wall patches over the same nodes, and one that shares an end node
    "shared": [dict(type=2, raw=(8, 20, 0, 0, 0, 0), label=2, t_wall=300.0, isothermal=True),
               dict(type=2, raw=(20, 33, 0, 0, 0, 0), label=2, t_wall=300.0, isothermal=True)],
    # a patch whose ghosts and interior reach into another's corner
    "corner": [dict(type=6, raw=(39, 39, 0, 6, 0, 0), label=6), dict(type=6, raw=(37, 39, 0, 0, 0, 0), label=6)],
}


@pytest.mark.parametrize("extra", sorted(EXTRA))
def test_ranges_that_meet(tmp_path, extra):
    case = cases.c1_case(40, 20)
    for b in case["bcs"]:
        if b["type"] == 2:
            for e in EXTRA[extra]:
                if e["type"] == 2:
                    e.update(t_wall=b.get("t_wall", 300.0), label=b["label"])
    case["bcs"] = case["bcs"] + EXTRA[extra]
    s = ostc.solver_for_case(case, str(tmp_path / extra))
    z = oracle_zone(case)
    s.step(6)
    z.run(6)
    errs = grouped(s.download("bv"), z.field("bv"), 6, BV_GROUPS)
    print(extra, {k: "%.1e" % v for k, v in errs.items()}, flush=True)
    assert max(errs.values()) < 1e-12 and np.all(np.isfinite(s.download("bv")))
