"""Counts and segments made on the device, at the edges of the cut.

- A grid without screening holds far more terms than the room first set aside
  for its segments, so the cut runs a second time with the room it asked for
  (a lost or doubled segment would change the values and the kernel's count).
- A batch whose applies hold very different counts, one with none.
Term counts equal the oracle's; FP64 values agree to 1e-12 of the largest as
in the other parity tests."""
import numpy as np
import pytest

import mrchem_amd as mw
import oracle

pytestmark = pytest.mark.gpu


def _mra(order):
    return mw.MultiResolutionAnalysis(order=order, min_scale=-4, scaling_factor=1.25, max_depth=8)


@pytest.mark.parametrize("order,mode", [(2, "fp64"), (2, "split16"), (4, "fp64")])
def test_more_segments_than_room(ctx, order, mode):
    mra = _mra(order)
    P = mw.PoissonOperator(mra, 1e-2)
    rho = mw.FunctionTree(mra).project_gaussians(1e-2, [1.0], [2.0], [[0.3, -0.2, 0.1]], max_depth=2)
    full = mw.FunctionTree(mra).project_gaussians(1e-12, [1.0], [0.02], [[0.0, 0.0, 0.0]], max_depth=1)
    d, l, _ = full.nodes()
    assert len(d) == 72
    out = mw.FunctionTree(mra).set_nodes(d, l)
    thr = np.zeros(len(d))
    plan = mw.ApplyPlan(out, P, rho, thr, mode=mode, ctx=ctx)
    ref, st = oracle.apply_fixed(mra, P.tables(), rho.nodes(), d, l, thr)
    info = plan.info()
    print("order %d %s: %d terms in %d segments" % (order, mode, st["term_apps"], info["segments"]))
    assert info["segments"] > (16384 + 64 * len(d) if mode == "fp64" else 2048 + 16 * len(d))
    r = plan.execute()
    assert r["term_apps"] == st["term_apps"] == info["host_term_apps"]
    plan.finish()
    # without a positive threshold every term is of the FP64 class
    assert np.max(np.abs(out.nodes()[2] - ref)) < 1e-12 * np.max(np.abs(ref))


@pytest.mark.parametrize("order,mode,prec,levels", [(2, "fp64", 1e-12, 1), (4, "fp64", 1e-12, 1),
                                                    (2, "mixed", 1e-30, 2), (2, "split16", 1e-30, 2)])
def test_adaptive_level_with_more_segments_than_room(order, mode, prec, levels):
    # an adaptive level starts its calculator before the host knows the
    # number of segments; here the last level needs more than its room
    mra = _mra(order)
    P = mw.PoissonOperator(mra, 1e-10)
    rho = mw.FunctionTree(mra).project_gaussians(1e-2, [1.0], [2.0], [[0.3, -0.2, 0.1]], max_depth=2)
    out = mw.FunctionTree(mra)
    ctx = mw.Context(0)
    ctx.set_precision(mode)
    mw.apply(prec, out, P, rho, max_iter=levels, abs_prec=True, ctx=ctx)
    stats = ctx.last_stats()
    d, l, c = out.nodes()
    thr = out.thresholds()
    od, ol, othr, oc, st = oracle.apply_adaptive(mra, P.tables(), rho.nodes(), prec, abs_prec=True, max_iter=levels,
                                                 max_depth=mra.max_depth)
    np.testing.assert_array_equal(d, od)
    np.testing.assert_array_equal(l, ol)
    # estimates at roundoff of so small a threshold may fall on either side
    assert abs(stats["term_apps"] - st["term_apps"]) < 1e-4 * st["term_apps"]
    n1 = int((d > 0).sum())
    # a low-precision term is off by at most 1e-3 of 16 thresholds
    low = 0.0 if mode == "fp64" else 16e-3 * np.max(thr) * st["term_apps"] / (8 * n1)
    assert np.max(np.abs(c - oc)) < 1e-12 * np.max(np.abs(oc)) + low
    plan = mw.ApplyPlan(mw.FunctionTree(mra).set_nodes(d, l), P, rho, thr, mode=mode, ctx=ctx)
    print("order %d: %d nodes, %d segments" % (order, n1, plan.info()["segments"]))
    room = 16384 + 64 * n1 if mode == "fp64" else levels * 2048 + 16 * n1  # of all levels but the roots
    assert plan.info()["segments"] > room
    assert plan.execute()["term_apps"] == stats["term_apps"]


@pytest.mark.parametrize("mode", ["fp64", "mixed"])
def test_batch_of_unequal_counts(ctx, mode):
    mra = _mra(3)
    P = mw.PoissonOperator(mra, 1e-2)
    f = mw.FunctionTree(mra).project_gaussians(1e-3, [1.0], [20.0], [[0.3, -0.2, 0.1]])
    g = mw.FunctionTree(mra).project_gaussians(1e-1, [1.0], [0.05], [[0.0, 0.5, 0.0]])
    outs, thrs = [], []
    for t, s in ((f, 1e-5), (g, 1e-2), (g, 1e6)):
        d, l, _ = t.nodes()
        outs.append(mw.FunctionTree(mra).set_nodes(d, l))
        thrs.append(np.full(len(d), s))
    inps = [f, g, g]
    plan = mw.ApplyPlan(outs, P, inps, thrs, mode=mode, ctx=ctx)
    r = plan.execute()
    plan.finish()
    total = 0
    for o, i, t in zip(outs, inps, thrs):
        d, l, c = o.nodes()
        ref, st = oracle.apply_fixed(mra, P.tables(), i.nodes(), d, l, t)
        total += st["term_apps"]
        assert np.max(np.abs(c - ref)) <= (1e-12 if mode == "fp64" else 1e-6) * max(np.max(np.abs(ref)), 1e-300)
    print("%s: %d terms" % (mode, total))
    assert r["term_apps"] == total == plan.info()["host_term_apps"] > 0
