"""Quotients and reciprocals of the reference form without IEEE divisions, at
the operands where such sequences go wrong; bit patterns against the oracle."""
import numpy as np
import pytest

import oracle as O
from sedcol import capi, cases

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.ascontiguousarray(a).view(np.int64)


def test_reciprocal_of_a_mantissa_of_ones(gpu_ready):
    """The pathway sum 1 - 2^-53: its reciprocal lies 2^-106 above the middle of
    two doubles, where a correction by the residual meets a tie."""
    dom = cases.plain_columns(ni=64, nj=1, K=16, seed=6)
    dom.params.kin.kinO2anox = 2.0 ** -50
    dom.params.kin.ksO2oxic = 3.0
    o2 = 3.0 * 2.0 ** 53
    assert o2 / (o2 + 3.0) == 1.0 - 2.0 ** -53
    rng = np.random.default_rng(1)
    x = dom.conc0.copy()
    x[:5] = 10.0 ** rng.uniform(0.0, 5.0, size=x[:5].shape)
    x[5] = o2
    x[6:9] = 0.0
    dom.cbw[0, 5] = o2
    p = dom.params.si()
    with capi.SedimentColumns.from_domain(dom) as g:
        rg, fg = g.get_rhs(x)
    ro, fo = O.Oracle(dom, p).rhs(x)
    assert np.array_equal(rg, ro) and np.array_equal(fg, fo)


@pytest.mark.parametrize("wide", [False, True])
def test_sign_of_zero(gpu_ready, wide):
    """No bioturbation and a given concentration at the top: the particulate
    fluxes are quotients of a zero of either sign."""
    dom = cases.plain_columns(ni=9, nj=1, K=15, seed=6)
    dom.biot[:] = 0.0
    dom.params.bcup_part = 2
    rng = np.random.default_rng(2)
    x = rng.uniform(0.0, 200.0, size=dom.conc0.shape)
    dom.cbw[0] = rng.uniform(0.0, 200.0, size=dom.cbw[0].shape)
    if wide:
        x[3, ::15] = 1.0e-200  # one value per column outside the fast range
    with capi.SedimentColumns.from_domain(dom) as g:
        rg, fg = g.get_rhs(x)
    ro, fo = O.Oracle(dom, dom.params.si()).rhs(x)
    assert np.any(_bits(fo[:5]) == 0) and np.any(_bits(fo[:5]) != 0)
    assert np.array_equal(_bits(fg), _bits(fo))
    assert np.array_equal(_bits(rg), _bits(ro))
