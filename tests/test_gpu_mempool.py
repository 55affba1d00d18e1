"""The contexts' device memory pools: two contexts working in two threads give
the results of a serial run, and a destroyed context gives its idle blocks
back to the driver."""
import ctypes
import gc
import threading

import numpy as np
import pytest

import mrchem_amd as mw

pytestmark = pytest.mark.gpu


def _work(ctx, mra, reps):
    prec = 1e-3
    P = mw.build_operators(mra, [0.0], prec, ctx=ctx)[0]
    f = mw.FunctionTree(mra).project_gaussians(prec, [1.0, 0.5], [8.0, 3.0], [[0.2, -0.3, 0.1], [-0.5, 0.4, 0.0]])
    out = []
    for _ in range(reps):
        V = mw.FunctionTree(mra).set_resident(ctx)
        mw.apply(prec, V, P, f, ctx=ctx)
        W = mw.multiply(prec, mw.FunctionTree(mra).set_resident(ctx), f, V, abs_prec=True, ctx=ctx)
        out.append((V.nodes(), W.nodes()))
    return out


def _free():
    """Free device bytes, from the HIP runtime the library is linked to."""
    free, total = ctypes.c_size_t(0), ctypes.c_size_t(0)
    assert mw.lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_two_contexts_in_threads_and_release():
    mra = mw.MultiResolutionAnalysis(order=5, max_depth=10, min_scale=-4, scaling_factor=1.25)
    serial = _work(mw.Context(0), mra, 1)[0]
    gc.collect()
    free0 = _free()
    ctxs = [mw.Context(0), mw.Context(0)]
    got = [None, None]

    def run(i):
        got[i] = _work(ctxs[i], mra, 4)

    th = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for g in got:
        for pair in g:
            for (d, l, c), (d0, l0, c0) in zip(pair, serial):
                assert np.array_equal(d, d0) and np.array_equal(l, l0)
                # sums of a node's segments are atomic: equal to rounding
                assert np.max(np.abs(c - c0)) < 1e-12 * np.max(np.abs(c0))
    held = free0 - _free()
    del ctxs, got, g, pair
    gc.collect()
    left = free0 - _free()
    print("pools held %.1f MB, %.1f MB after the contexts' end" % (held / 1e6, left / 1e6))
    assert held > 0 and left <= held / 4
