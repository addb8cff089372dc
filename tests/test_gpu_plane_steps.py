"""2-D blocks: what a call leaves behind does not depend on how the steps are
cut into calls, although the k-ghost planes are written by a call's last stage
alone and the time step of a stage comes out of the stage before it."""
import numpy as np
import pytest

import ostc
from ostc import cases

pytestmark = pytest.mark.gpu

# vel and mach on the ghost planes are what the boundary ranges derive there
# from the planes that a stage before left
FIELDS = ("bv", "sv", "cv", "dq", "vel", "mach", "acoustic", "mul", "cond", "gamma", "cp", "rhoD", "mut", "turb_cond",
          "dt_local")


def _case(kind, size):
    if kind in ("mixing", "farfield"):
        case = cases.c3_case(*size)
        if kind == "farfield":
            case["setup"]["array string boundary_conditions"] = ["air_stream", "fuel_stream", "outflow", "farfield"]
            case["setup"]["struct farfield"] = [
                ("string", "type", "farfield"), ("int", "label", 4), ("real", "mach", 2.0),
                ("real", "pressure", 101325.0), ("real", "temperature", 1500.0), ("real", "u", 1.0),
                ("real", "v", 0.0), ("real", "w", 0.0), ("real", "O2", 0.233), ("real", "N2", 0.767)]
            for b in case["bcs"]:
                if b["type"] == 3:
                    b["type"], b["label"] = 4, 4
        return case
    if kind == "plate":
        return cases.sst_plate_case(*size)
    case = cases.c1_case(*size)
    if kind == "fixed":
        case["setup"]["bool fixed_time_step"], case["setup"]["real dt"] = 1, 2e-7
    if kind == "inside":  # a symmetry patch on a layer inside the block
        case["bcs"].append(dict(type=3, raw=(30, 30, 8, 20, 0, 0), label=3))
    return case


def _solver(kind, size, root):
    case = _case(kind, size)
    if case["name"] == "c1":
        return case, ostc.solver_for_case(case, root)
    s = ostc.solver_for_case(case, root, initial=False)
    if case["name"] == "c3":
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
@pytest.mark.parametrize("kind,size", [("air", (12, 12)), ("air", (62, 37)), ("air", (513, 511)), ("fixed", (62, 37)),
                                       ("inside", (62, 37)), ("mixing", (33, 17)), ("farfield", (33, 17)),
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


@pytest.mark.parametrize("kind,size", [("air", (62, 37)), ("inside", (62, 37)), ("mixing", (33, 17)),
                                       ("farfield", (33, 17)), ("plate", (60, 40))])
def test_stage_by_stage(tmp_path, kind, size):
    """A call of several steps leaves what its stages leave when each is asked
    for by itself, with the boundary ranges on every plane: the same kernels on
    the same values, so nothing differs but where a sum is contracted."""
    case, s = _solver(kind, size, str(tmp_path / "call"))
    _, t = _solver(kind, size, str(tmp_path / "stages"))
    s.step(3)
    for _ in range(3):
        for rk in range(3):
            t.rhs()
            dt = t.global_dt()
            t.rk3_stage(dt, rk)
            t.apply_bc(True)
            t.update_properties()
    for f in FIELDS:
        a, b = s.download(f), t.download(f)
        assert np.array_equal(np.isnan(a), np.isnan(b)), f
        if a.size:
            scale = max(np.nanmax(np.abs(b)), 1e-300)
            assert np.nanmax(np.abs(a - b)) <= 1e-13 * scale, (f, np.nanmax(np.abs(a - b)) / scale)
