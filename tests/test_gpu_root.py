"""The root level's dense kernels against the oracle, over tile widths and worlds.

An apply stopped after its first level (max_iter = 0) computes the root boxes
alone, with threshold zero, so every term of every box pair and component is
applied.  A root value is a sum of at most M (2 N b)^3 FP64 products in
another order than the oracle's; with rounding errors that do not line up it
stays within sqrt(1e7) 2^-53 ~ 4e-13 of the largest value, so 1e-12 holds it.
"""
import numpy as np
import pytest

import mrchem_amd as mw
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,corner,boxes,basis", [
    (1, (0, 0, 0), (1, 1, 1), "interpolating"),     # 4 of 16 values a direction
    (7, (0, 0, 0), (1, 1, 1), "interpolating"),     # one whole tile
    (4, (-1, -1, -1), (2, 2, 2), "legendre"),       # 20 of 32
    (7, (-1, -1, -1), (2, 2, 2), "interpolating"),  # two whole tiles
    (10, (-1, -1, -1), (2, 2, 2), "interpolating"),  # 44 of 48
    (11, (-1, -1, -1), (2, 2, 2), "interpolating"),  # three whole tiles
    (5, (-1, 0, -1), (2, 1, 2), "interpolating"),   # a matrix per direction
    (8, (0, -1, 0), (1, 2, 1), "interpolating"),
    (11, (-1, -1, 0), (2, 2, 1), "interpolating"),
])
def test_root_level(ctx, order, corner, boxes, basis):
    mra = mw.MultiResolutionAnalysis(order=order, basis=basis, min_scale=-2, corner=corner, boxes=boxes, max_depth=8)
    prec = 1e-3
    P = mw.PoissonOperator(mra, prec)
    lo = np.array(corner) * 4.0
    cen = lo + 4.0 * np.array(boxes) * np.array([[0.41, 0.63, 0.37], [0.72, 0.28, 0.55]])
    rho = mw.FunctionTree(mra).project_gaussians(prec, [1.0, -0.6], [0.9, 2.0], cen)
    V = mw.FunctionTree(mra)
    mw.apply(prec, V, P, rho, max_iter=0, ctx=ctx)
    od, ol, oc = V.nodes()
    assert len(od) == np.prod(boxes) and not np.any(V.thresholds())
    ref, st = oracle.apply_fixed(mra, P.tables(), rho.nodes(), od, ol, V.thresholds())
    err = np.max(np.abs(ref - oc)) / np.max(np.abs(ref))
    print("order %d boxes %s: %d terms, error %.2e" % (order, boxes, st["term_apps"], err))
    assert err < 1e-12
    assert ctx.last_stats()["term_apps"] == st["term_apps"]
    # a frozen plan in the split mode classes the roots' terms by bound when
    # another threshold is positive, and takes them in FP64 when none is
    for thr in (np.zeros(len(od)), np.where(np.arange(len(od)) == 0, 1e-9, 0.0)):
        plan = mw.ApplyPlan(V, P, rho, thr, mode="split16", ctx=ctx)
        r = plan.execute()
        want, ws = oracle.apply_fixed(mra, P.tables(), rho.nodes(), od, ol, thr)
        assert r["term_apps"] == ws["term_apps"]
        plan.finish()
        err = np.max(np.abs(V.nodes()[2] - want)) / np.max(np.abs(want))
        assert err < (1e-12 if not thr.any() else 1e-6)
        del plan
