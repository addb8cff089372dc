"""GPU Newton temperature (one mixture polynomial per species-branch interval)
against the CPU oracle's species-by-species inversion, where the branches
change: below and at t_low (200 and 300 K), around t_mid (1000 K), and warm
starts on the other side of a branch point."""
import numpy as np
import pytest

import pyoracle as po
from test_gpu_mixture import NS, _setup

pytestmark = pytest.mark.gpu

TRUE_T = [150.0, 199.9, 200.0, 200.1, 299.9, 300.0, 305.0, 700.0, 999.0, 999.9999, 1000.0, 1000.0001, 1001.0, 1500.0,
          2900.0]
WARM = [1.0, 1.0005, 0.8, 1.3, 0.99, 1.01]


@pytest.mark.parametrize("warm", WARM)
def test_newton_temperature_at_branch_points(tmp_path, mech, warm):
    case, s, _, _ = _setup(tmp_path, mech)
    g, mx, my = case["ngg"], case["mx"], case["my"]
    shape = (1 + 2 * g, my + 2 * g, mx + 2 * g)
    bv = s.download("bv").reshape((6,) + shape)
    sv = s.download("sv").reshape((NS,) + shape)
    rng = np.random.default_rng(11)
    Y = rng.random((NS, my, mx)) + 1e-3
    Y[1, ::2] = 0.0  # absent species
    Y /= Y.sum(axis=0)
    T = np.resize(np.array(TRUE_T), my * mx).reshape(my, mx)
    at = (g, slice(g, g + my), slice(g, g + mx))
    mw = np.array([mech.mw[i] for i in range(NS)])
    sv[(slice(None),) + at] = Y
    bv[(5,) + at] = T
    bv[(4,) + at] = 1e5
    bv[(0,) + at] = 1e5 / (8314.462618 * T * (Y / mw[:, None, None]).sum(axis=0))
    s.upload("bv", bv)
    s.upload("sv", sv)
    s.initialize()
    cv = s.download("cv").reshape((5 + NS,) + shape)
    start = s.download("bv").reshape((6,) + shape)
    start[5] *= warm
    s.upload("bv", start)
    n, _, _ = s.field_info("dq")
    s.upload("dq", np.zeros(n))
    s.rk3_stage(1e-9, 0)
    got = s.download("bv").reshape((6,) + shape)
    worst = 0.0
    for j in range(g, g + my):
        for i in range(g, g + mx):
            q = cv[:, g, j, i]
            vel = np.array([q[1], q[2], 0.0]) / q[0]  # the 2-D stage drops rho w
            want = po.temperature_newton(mech, q[0], q[4], vel, q[5:] / q[0], start[5, g, j, i])[0]
            worst = max(worst, abs(got[5, g, j, i] - want) / want)
    print("warm start x%.4f: worst relative T error %.2e" % (warm, worst), flush=True)
    # e has relative rounding of a few ulp; de/dT = cv and |e| up to about
    # 50 cv T (formation enthalpies) leave about 1e-14 of T
    assert worst < 1e-12
    s.close()
