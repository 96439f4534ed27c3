"""States of the transposed layout on both sides of the sizes up to which the host
transposes them: round trip and right-hand side, also over its own input."""
import numpy as np
import pytest

import oracle as O
from sedcol import capi, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncol,K", [(1, 1), (7, 64), (1100, 5), (1101, 5), (1000, 7), (1001, 7), (4000, 24)])
def test_round_trip_and_rhs(gpu_ready, ncol, K):
    dom = cases.plain_columns(ni=ncol, nj=1, K=K, seed=5)
    rng = np.random.default_rng(ncol)
    x, y = rng.uniform(0.1, 100.0, (2, 11, K, ncol))
    ro, fo = O.Oracle(dom, dom.params.si()).rhs(dom.packed_state(x))
    with capi.SedimentColumns(dom.nlayers, dom.mask, layout="fortran") as g:
        g.set_params(dom.params)
        g.set_geometry(*[a.reshape(ncol, K).T for a in (dom.dz, dom.dzc, dom.phi, dom.phiI, dom.bfac)], dom.biot)
        g.set_forcing(*dom.record(0))
        g.set_state(y)
        rg, fg = g.get_rhs(x)
        assert np.array_equal(g.get_state(), y)  # the right-hand side leaves the state alone
        assert np.array_equal(dom.packed_state(rg), ro) and np.array_equal(fg, fo)
        z = x.copy()
        capi.check(capi.lib().sedcol_rhs(g._h, capi._pd(z), capi._pd(z), None))
        assert np.array_equal(z, rg)
