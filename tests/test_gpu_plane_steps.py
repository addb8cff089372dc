"""2-D blocks: what a call leaves behind does not depend on how the steps are
cut into calls, although the k-ghost planes are written by a call's last stage
alone and the time step of a stage comes out of the stage before it."""
import numpy as np
import pytest

import ostc
from ostc import cases

pytestmark = pytest.mark.gpu

FIELDS = ("bv", "sv", "cv", "dq", "acoustic", "mul", "cond", "dt_local")


def _solver(kind, size, root):
    case = {"air": cases.c1_case, "mixing": cases.c3_case, "plate": cases.sst_plate_case}[kind](*size)
    if kind == "air":
        return case, ostc.solver_for_case(case, root)
    s = ostc.solver_for_case(case, root, initial=False)
    if kind == "mixing":
        st = {}
        for k in ("air_stream", "fuel_stream"):
            o = s.inflow_state(k, 16)
            st[k] = dict(rho=o[0], u=o[1], v=o[2], w=o[3], p=o[4], t=o[5], vel=o[6], sv=o[7:16])
        bv, sv = cases.c3_fields(case, st, s.table("mw", 9))
    else:
        bv, sv = cases.sst_plate_fields(case)
    s.upload("bv", bv)
    s.upload("sv", sv)
    s.initialize()
    return case, s


# 14 x 14 points with ghosts are less than one workgroup, 513 x 511 need more
# than the 1024 partial minima that the update reduces itself
@pytest.mark.parametrize("kind,size", [("air", (12, 12)), ("air", (62, 37)), ("air", (513, 511)), ("mixing", (33, 17)),
                                       ("plate", (60, 40))])
def test_calls_cut_differently(tmp_path, kind, size):
    out = []
    for n, cuts in enumerate(((4,), (1, 2, 1), (1, 1, 1, 1))):
        case, s = _solver(kind, size, str(tmp_path / str(n)))
        dts = np.concatenate([s.step(c)[0] for c in cuts])
        out.append((dts, {f: np.array(s.download(f)) for f in FIELDS}))
    g = case["ngg"]
    for dts, fields in out[1:]:
        assert np.array_equal(dts, out[0][0])
        for f in FIELDS:
            assert np.array_equal(fields[f], out[0][1][f], equal_nan=True), f
    for f in ("bv", "sv", "cv"):
        a = out[0][1][f]
        if a.size:
            a = a.reshape((-1,) + cases.ghost_shape(case["mx"], case["my"], case["mz"], g))
            assert all(np.array_equal(a[:, k], a[:, g]) for k in range(2 * g + 1)), f
