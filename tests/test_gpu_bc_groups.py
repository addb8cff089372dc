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
    # an outflow patch on the lower symmetry face: outflow ranges go first, the
    # symmetry then overwrites what both write
    "overlap": [dict(type=6, raw=(5, 12, 0, 0, 0, 0), label=6)],
    # a cold and a hot wall on the lower face, in this order, that share nodes
    # 14 to 20: the hot one has the last word there
    "shared": [dict(type=2, raw=(8, 20, 0, 0, 0, 0), label=20, t_wall=250.0, isothermal=True),
               dict(type=2, raw=(14, 33, 0, 0, 0, 0), label=21, t_wall=900.0, isothermal=True)],
    # a patch whose ghosts and interior reach into another's corner
    "corner": [dict(type=6, raw=(39, 39, 0, 6, 0, 0), label=6), dict(type=6, raw=(37, 39, 0, 0, 0, 0), label=6)],
}


@pytest.mark.parametrize("extra", sorted(EXTRA))
def test_ranges_that_meet(tmp_path, extra):
    case = cases.c1_case(40, 20)
    walls = [b for b in EXTRA[extra] if b["type"] == 2]
    for b in walls:
        name = "wall%d" % b["label"]
        case["setup"]["array string boundary_conditions"].append(name)
        case["setup"]["struct " + name] = [("string", "type", "wall"), ("int", "label", b["label"]),
                                           ("string", "thermal_type", "isothermal"),
                                           ("real", "temperature", b["t_wall"])]
    case["bcs"] = case["bcs"] + EXTRA[extra]
    s = ostc.solver_for_case(case, str(tmp_path / extra))
    z = oracle_zone(case)
    s.step(6)
    z.run(6)
    errs = grouped(s.download("bv"), z.field("bv"), 6, BV_GROUPS)
    print(extra, {k: "%.1e" % v for k, v in errs.items()}, flush=True)
    assert max(errs.values()) < 1e-12 and np.all(np.isfinite(s.download("bv")))
    if walls:
        t = s.download("bv").reshape((6,) + cases.ghost_shape(case["mx"], case["my"], case["mz"], case["ngg"]))[5]
        g = case["ngg"]
        assert t[g, g, g + 10] == 250.0 and t[g, g, g + 17] == 900.0
