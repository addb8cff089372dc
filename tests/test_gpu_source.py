"""The finite-rate source and its Jacobian on a flow block against the oracle,
for every way the kinetics loop walks a reaction."""
import os
import shutil

import numpy as np
import pytest

import ostc
import pyoracle as po
from ostc import cases
from helpers import grouped, oracle_zone, relerr

pytestmark = pytest.mark.gpu

NS = 9
# forms the mechanism file lacks: three molecules on a side, a species on
# both sides (here the bath gas, which is then not inert), more than four
# species, irreversible, and explicit reverse rates
FORMS = """H2+H2+O2=H2O+H2O  1.0E+14  0.00  2.0E+04
O2+N2=O+O+N2  1.0E+16  -0.50  1.18E+05
H2+O2=>OH+OH  1.7E+13  0.00  4.8E+04
H2O2+H2=H2O+H+OH  2.0E+13  0.00  2.0E+04
HO2+H2=H2O2+H  3.0E+13  0.00  2.4E+04
  REV/ 4.82E+13 0.00 7.95E+03 /
"""


def _tables(s):
    nr = s.get_int("n_reac")
    t = {k: s.table(k, 63) for k in ("high_coeff", "low_coeff")}
    t.update({k: s.table(k, 81) for k in ("WjDivWi_to_One4th", "sqrt_WiDivWjPl1Mul8", "binary_diffusivity_coeff",
                                         "kb_over_eps_jk")})
    t.update({k: s.table(k, NS) for k in ("mw", "t_low", "t_mid", "t_high", "LJ_potent_inv", "vis_coeff")})
    t.update({k: s.table(k, nr) for k in ("label", "order", "A", "b", "Ea", "A2", "b2", "Ea2", "troe_alpha",
                                         "troe_t3", "troe_t1", "troe_t2")})
    t.update({k: s.table(k, nr * NS) for k in ("stoi_f", "stoi_b", "third_body_coeff")})
    t.update(n_spec=NS, n_reac=nr)
    return t


@pytest.mark.parametrize("method", [0, 1, 2])
@pytest.mark.parametrize("bath", [False, True])
@pytest.mark.parametrize("cold", [False, True])
def test_source_reaction_forms(tmp_path, method, bath, cold):
    """Explicit, exact-point-implicit and diagonal source, with the bath gas
    inert (left out of the Jacobian's sums) and reacting, at flame
    temperatures and across the lower end of the thermodynamic fits.  The
    species rows and the Jacobian are held to 1e-12 of their largest entry:
    the exponentials' arguments reach 200, each rounded to 200 x 2^-53."""
    case = cases.c3_case(23, 11)  # 253 cells: a partial last workgroup
    case["setup"]["int chemSrcMethod"] = method
    case["scheme"] = dict(case["scheme"], chemSrcMethod=method)
    root = str(tmp_path / "forms")
    chem = os.path.join(root, "input_files", "chemistry")
    shutil.copytree(cases.CHEM_DIR, chem)
    path = os.path.join(chem, "combustion_mechanism.inp")
    text = open(path).read().rstrip()
    assert text.endswith("END")
    with open(path, "w") as f:
        f.write(text[:-3] + "".join(ln for ln in FORMS.splitlines(keepends=True) if bath or "N2" not in ln) + "END\n")
    s = ostc.solver_for_case(case, root, initial=False)
    mech = po.make_mech(_tables(s))
    states = {}
    for name in ("air_stream", "fuel_stream"):
        o = s.inflow_state(name, 7 + NS)
        states[name] = dict(rho=o[0], u=o[1], v=o[2], w=o[3], p=o[4], t=o[5], vel=o[6], sv=o[7:7 + NS])
    for b in case["bcs"]:
        if b["type"] == 5:
            b["state"] = states[b["stream"]]
    mw = np.array([mech.mw[i] for i in range(NS)])
    bv, sv = cases.c3_fields(case, states, mw)
    rng = np.random.default_rng(5)
    for l in (1, 3, 4, 5, 6, 7):  # radicals and products
        sv[l] = 10.0 ** rng.uniform(-6, -2, sv[l].shape)
    sv /= sv.sum(axis=0)
    bv[5] = rng.uniform(200.0, 320.0, bv[5].shape) if cold else rng.uniform(900.0, 2400.0, bv[5].shape)
    bv[0] = bv[4] / (8314.462618 * bv[5] * np.tensordot(1 / mw, sv, axes=(0, 0)))
    s.upload("bv", bv)
    s.upload("sv", sv)
    s.initialize()
    z = oracle_zone(case, mech=mech, bv=bv, sv=sv)
    s.rhs()
    z.rhs()
    errs = grouped(s.download("dq"), z.field("dq"), 14, {"flow": range(5), "species": range(5, 14)})
    if method:
        n = s.download("chem_jac").size
        errs["jac"] = relerr(s.download("chem_jac"), z.field("chem_jac")[:n])
    print("source method=%d bath=%d cold=%d nr=%d" % (method, bath, cold, mech.n_reac),
          {k: "%.2e" % v for k, v in errs.items()}, flush=True)
    assert max(errs.values()) < 1e-12
