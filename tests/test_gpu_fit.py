"""Kernel fits of device-built operators: the step size chosen from errors
evaluated on the device is the one the host search takes, so the terms are the
same to the bit.  The reported errors are sums of at most 300 positive terms
of total 1 with two different exp: within 300 x 2^-53 + 2^-52 of each other,
held to 1e-13.  A kernel that no step fits is refused by both."""
import numpy as np
import pytest

import mrchem_amd as mw

pytestmark = pytest.mark.gpu


def _mra(order):
    return mw.MultiResolutionAnalysis(order=order, min_scale=-4, scaling_factor=1.25, max_depth=10)


@pytest.mark.parametrize("order,prec", [(2, 1e-2), (4, 1e-4), (7, 1e-6), (11, 1e-7)])
def test_fits_equal_the_host_search(ctx, order, prec):
    mra = _mra(order)
    mus = [0.0, 0.05, 0.7, 2.5]
    for mu, dev in zip(mus, mw.build_operators(mra, mus, prec, ctx=ctx)):
        host = mw.HelmholtzOperator(mra, mu, prec) if mu else mw.PoissonOperator(mra, prec)
        (a, b), (a0, b0) = dev.terms(), host.terms()
        assert len(a) <= 300 and np.array_equal(a, a0) and np.array_equal(b, b0)
        e, e0 = dev.info()["fit_err"], host.info()["fit_err"]
        assert abs(e - e0) < 1e-13 and 0 < e <= prec / 20


def test_a_kernel_that_is_not_fitted(ctx):
    mra = _mra(4)
    with pytest.raises(mw.MWGError, match="accuracy not reached"):
        mw.HelmholtzOperator(mra, 9.0, 1e-4)
    with pytest.raises(mw.MWGError, match="accuracy not reached"):
        mw.build_operators(mra, [0.5, 9.0], 1e-4, ctx=ctx)
