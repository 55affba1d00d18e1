"""Bands and input slots found on the device, where the search can go wrong:

- an input far shallower than the output grid, so that slots are generated
  through chains of generated ancestors, some of which are slots of coarser
  output nodes themselves;
- the opposite, an input far deeper than the grid;
- several applies with the same and with different inputs in one plan;
- one, four and eight root boxes, output nodes at the edge of the world.
Slots, generated slots and terms are counted by the oracle; values agree with
it to 1e-12 of the largest, as in the other parity tests."""
import numpy as np
import pytest

import mrchem_amd as mw
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("corner,boxes", [((-1, -1, -1), (2, 2, 2)), ((0, 0, 0), (1, 1, 1)), ((-1, 0, -1), (2, 1, 2))])
@pytest.mark.parametrize("deep", ["out", "inp"])
def test_chains_of_generated_nodes(ctx, corner, boxes, deep):
    mra = mw.MultiResolutionAnalysis(order=3, min_scale=-4, corner=corner, boxes=boxes, scaling_factor=1.0,
                                     max_depth=9)
    P = mw.PoissonOperator(mra, 1e-3)
    # beside the origin, a corner of the one-box world
    sharp = mw.FunctionTree(mra).project_gaussians(1e-3, [1.0], [4e3], [[0.4, 0.3, 0.2]])
    wide = mw.FunctionTree(mra).project_gaussians(1e-1, [1.0], [0.3], [[1.0, 2.0, 1.0]], max_depth=1)
    inp, grid = (wide, sharp) if deep == "out" else (sharp, wide)
    d, l, _ = grid.nodes()
    out = mw.FunctionTree(mra).set_nodes(d, l)
    thr = np.where(d == 0, 0.0, 1e-7)
    plan = mw.ApplyPlan(out, P, inp, thr, ctx=ctx)
    ref, st = oracle.apply_fixed(mra, P.tables(), inp.nodes(), d, l, thr)
    info = plan.info()
    r = plan.execute()
    plan.finish()
    print("depths %d and %d: %d slots, %d generated" % (d.max(), inp.nodes()[0].max(), info["in_slots"], info["generated"]))
    assert r["term_apps"] == st["term_apps"]
    assert info["in_slots"] == st["slots"] and info["generated"] == st["generated"]
    assert np.max(np.abs(out.nodes()[2] - ref)) < 1e-12 * np.max(np.abs(ref))


def test_applies_of_shared_and_distinct_inputs(ctx):
    mra = mw.MultiResolutionAnalysis(order=4, min_scale=-4, scaling_factor=1.25, max_depth=9)
    P = mw.PoissonOperator(mra, 1e-3)
    f = mw.FunctionTree(mra).project_gaussians(1e-3, [1.0], [60.0], [[0.3, -0.2, 0.1]])
    g = mw.FunctionTree(mra).project_gaussians(1e-2, [1.0], [2.0], [[-1.0, 0.5, 0.0]])
    inps, grids = [f, g, f, g], [g, f, f, g]
    outs, thrs = [], []
    for t in grids:
        d, l, _ = t.nodes()
        outs.append(mw.FunctionTree(mra).set_nodes(d, l))
        thrs.append(np.where(d == 0, 0.0, 1e-6))
    plan = mw.ApplyPlan(outs, P, inps, thrs, ctx=ctx)
    info = plan.info()
    plan.execute()
    plan.finish()
    slots = gen = 0
    for o, i, t in zip(outs, inps, thrs):
        d, l, c = o.nodes()
        ref, st = oracle.apply_fixed(mra, P.tables(), i.nodes(), d, l, t)
        slots += st["slots"]
        gen += st["generated"]
        assert np.max(np.abs(c - ref)) < 1e-12 * np.max(np.abs(ref))
    assert (info["in_slots"], info["generated"]) == (slots, gen)
