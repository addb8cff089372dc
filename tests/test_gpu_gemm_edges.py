"""Loss and gradient of the network at batch sizes that leave the matrix
kernels partial tiles, K steps and split shares, against the numpy network
with BF16 operands."""
import numpy as np
import pytest

import mlp_oracle as mo
import ostc
from ostc import cases
from helpers import relerr

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def solver(tmp_path_factory):
    case = cases.c3_case(16, 8)
    root = str(tmp_path_factory.mktemp("gemm"))
    cases.write_case_dir(case, root)
    s = ostc.Solver(root, 0)
    s.surrogate_init(3)
    return s


# 8: one 8-row step; 56, 72: below and above a tile of 64; 264: a fifth K step
# of 8 rows in the one share; 1000: three shares, the last one partial; 8192:
# the 25 shares asked for are 21 of 384 rows and one of 128
@pytest.mark.parametrize("batch", [8, 56, 72, 264, 1000, 8192])
def test_gradient_batch_sizes(solver, batch):
    rng = np.random.default_rng(batch)
    p = mo.pack([(W, 0.1 * rng.standard_normal(b.shape)) for W, b in mo.unpack(mo.init_params(8))]).astype(np.float32)
    solver.surrogate_set_params(p)
    x = rng.standard_normal((batch, 11)).astype(np.float32)
    t = rng.standard_normal((batch, 8)).astype(np.float32)
    g, loss = solver.surrogate_gradient(x, t)
    lb, gb = mo.loss_and_grad(p.astype(float), x.astype(float), t.astype(float), bf=True)
    # FP32 sums of BF16 products in another order, which moves some of the
    # stored activations by one BF16 step (2^-9 relative)
    assert abs(loss - lb) <= 1e-5 * lb
    errs = [relerr(a, b) for (a, _), (b, _) in zip(mo.unpack(g), mo.unpack(gb))]
    errs += [relerr(a, b) for (_, a), (_, b) in zip(mo.unpack(g), mo.unpack(gb))]
    print("batch", batch, ["%.1e" % e for e in errs], flush=True)
    assert max(errs) < 2e-3
