"""Worlds far from the origin: a node's absolute translations, corner x 2^depth
and up, pass 32 bits there.

The plan of an apply and the results of applies, sums and products depend on
where nodes lie in the world alone, so a tree moved with its world to a corner
of 200,000 boxes gives the moved tree of the same results: the same grid, and
blocks to 1e-13 of the largest (a node's segments are added in no fixed order;
products and sums are equal to the bit)."""
import os
import subprocess

import numpy as np
import pytest

import mrchem_amd as mw

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NEAR, FAR = (-1, 0, -1), (200000, -300001, 2 ** 30)


def test_plans_do_not_depend_on_the_corner(tmp_path):
    csrc = os.path.join(ROOT, "mrchem_amd", "csrc")
    exe = str(tmp_path / "far_plan")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fopenmp", "-I" + csrc,
                    os.path.join(ROOT, "tests", "cxx", "far_plan.cpp")] +
                   [os.path.join(csrc, s) for s in ("mw_math.cpp", "mw_kernel.cpp", "mw_operator.cpp", "mw_tree.cpp",
                                                    "mw_plan.cpp")] + ["-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    print(r.stdout)
    assert r.returncode == 0, r.stdout


def _worlds(order):
    return [mw.MultiResolutionAnalysis(order=order, min_scale=-4, corner=c, boxes=(2, 2, 2), scaling_factor=1.25,
                                       max_depth=14) for c in (NEAR, FAR)]


def _moved_nodes(mra, tree):
    """The nodes of a tree, moved with its world's corner to that of mra."""
    d, l, c = tree.nodes()
    shift = np.array(mra.corner, dtype=np.int64) - np.array(tree.mra.corner, dtype=np.int64)
    return d, l + (shift[None] << d[:, None].astype(np.int64)), c


def _moved(mra, tree):
    return mw.FunctionTree(mra).set_nodes(*_moved_nodes(mra, tree))


def _same(near_tree, far_tree, tol):
    want = _moved_nodes(far_tree.mra, near_tree)
    d, l, c = far_tree.nodes()
    assert np.array_equal(d, want[0]) and np.array_equal(l, want[1])
    assert np.abs(l).max() > 2 ** 31
    assert np.max(np.abs(c - want[2])) <= tol * np.max(np.abs(want[2]))


def _inputs(near):
    """Sums of Gaussians of one centre, equal norms and exponents up to the given one."""
    out = []
    for top in (4e4, 6.0):
        a = top / 16.0 ** np.arange(4)
        out.append(mw.FunctionTree(near).project_gaussians(1e-2, a ** -0.75, a, [[11.3, 25.7, -2.1]] * 4))
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["fp64", "mixed", "split16"])
def test_apply_in_a_far_world(mode):
    ctx = mw.Context(0)
    ctx.set_precision(mode)
    got = []
    near, far = _worlds(3)
    inp = _inputs(near)[0]
    for mra in (near, far):
        f = _moved(mra, inp)
        V = mw.FunctionTree(mra)
        mw.apply(1e-3, V, mw.PoissonOperator(mra, 1e-3), f, ctx=ctx)
        got.append((V, ctx.last_stats()["term_apps"]))
    assert got[0][1] == got[1][1] > 0
    # the low-precision classes sum a segment in 32 bits, in no fixed cut
    _same(got[0][0], got[1][0], 1e-13 if mode == "fp64" else 1e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("resident", [False, True])
def test_sum_and_product_in_a_far_world(ctx, resident):
    got = []
    near, far = _worlds(3)
    for mra in (near, far):
        f, g = [_moved(mra, t) for t in _inputs(near)]
        out = [mw.FunctionTree(mra) for _ in range(3)]
        for t in [f, g] + out if resident else ():
            t.set_resident(ctx)
        mw.add(-1.0, out[0], [1.5, -0.25], [f, g], ctx=ctx)
        mw.multiply(1e-3, out[1], f, g, coef=1.3, max_iter=0, ctx=ctx)
        mw.add(-1.0, out[2], [1.0], [f], ctx=ctx)
        out[2].add(0.5, g, ctx=ctx)
        got.append(out)
    for a, b in zip(*got):
        _same(a, b, 0.0)
