"""Quotients of the reference form without IEEE divisions, at the operands where
such sequences go wrong; bit patterns against the oracle."""
import numpy as np
import pytest

import oracle as O
from sedcol import capi, cases

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.ascontiguousarray(a).view(np.int64)


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
