"""sedcol_step of a packed domain without land: the step's kernel takes the state
from the pinned memory of the call and leaves it there, in one launch per bin."""
import numpy as np
import pytest

import oracle as O
from sedcol import capi, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ni,nj,K", [(1, 2, 15), (4, 4, 16), (5, 3, 17), (73, 5, 15), (3, 2, 64)])
@pytest.mark.parametrize("method", [0, 1, 3, 4, 5])
def test_wet_step_bitwise(gpu_ready, ni, nj, K, method):
    dom = cases.plain_columns(ni=ni, nj=nj, K=K, seed=5)
    orc = O.Oracle(dom, dom.params.si())
    x, xo = dom.conc0.copy(), dom.conc0.copy()
    with capi.SedimentColumns.from_domain(dom) as g:
        for _ in range(3):
            f = g.ode_solver(x, 60.0, method)
            assert orc.ode_solver(xo, 60.0, method) == 0
            assert np.array_equal(x, xo) and np.array_equal(f, orc.flux)
        assert np.array_equal(g.get_state(), x)
        # the device's own copy goes on from there
        g.run(60.0, 2, method)
        for _ in range(2):
            assert orc.ode_solver(xo, 60.0, method) == 0
        assert np.array_equal(g.get_state(), xo)
        # a NaN is an error of this step alone
        y = x.copy()
        y[5, 3] = np.nan
        with pytest.raises(capi.SedcolError) as e:
            g.ode_solver(y, 60.0, method)
        assert e.value.code == capi.SEDCOL_ENAN
        g.ode_solver(x, 60.0, method)
