"""Input pools made on the device: generated input nodes several levels below
the input's finest nodes, and the slots' norms, against the oracle.

The output grid is refined where the input is not, so most band nodes are
generated, some as children of generated nodes.  Equal term counts pin the
norms of the slots (the screening reads them), equal blocks their values;
both sides are FP64 sums in different orders, so they agree to 1e-12 of the
largest value as in the other parity tests."""
import numpy as np
import pytest

import mrchem_amd as mw
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11])
def test_generated_inputs(ctx, order):
    mra = mw.MultiResolutionAnalysis(order=order, min_scale=-4, scaling_factor=1.25, max_depth=8)
    H = mw.HelmholtzOperator(mra, 1.0, 1e-3)
    rho = mw.FunctionTree(mra).project_gaussians(1e-1, [1.0, -0.4], [0.4, 0.7], [[0.3, -0.2, 0.1], [1.5, 0.4, -0.9]],
                                                 max_depth=3)
    grid = mw.FunctionTree(mra).project_gaussians(1e-2, [1.0], [60.0], [[0.31, 0.17, -0.22]], max_depth=5)
    d, l, _ = grid.nodes()
    out = mw.FunctionTree(mra).set_nodes(d, l)
    assert d.max() >= rho.nodes()[0].max() + 1
    thr = np.full(len(d), 1e-5 * rho.norm())
    plan = mw.ApplyPlan(out, H, rho, thr, ctx=ctx)
    r = plan.execute()
    assert plan.info()["generated"] > 20
    plan.finish()
    ref, st = oracle.apply_fixed(mra, H.tables(), rho.nodes(), d, l, thr)
    err = np.max(np.abs(out.nodes()[2] - ref)) / np.max(np.abs(ref))
    print("order %d: %d outputs, %d generated inputs, %d terms, error %.2e" %
          (order, len(d), plan.info()["generated"], st["term_apps"], err))
    assert r["term_apps"] == st["term_apps"] > 0
    assert err < 1e-12
