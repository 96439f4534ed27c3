"""Adaptive Euler beyond one workgroup, with a smallest step that is taken whether
or not the relative-change test passes: the failed test of the last attempt is
not an error; bitwise against the oracle."""
import numpy as np
import pytest

import oracle as O
from sedcol import capi, cases
from sedcol.params import ADAPTIVE_EULER

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ni,K", [(40, 30), (70, 16), (9, 64)])
@pytest.mark.parametrize("dt_min", [50.0, 1000.0])
def test_forced_steps_are_not_errors(gpu_ready, ni, K, dt_min):
    dom = cases.plain_columns(ni=ni, nj=1, K=K, seed=4)
    dom.params.dt_min = dt_min
    dom.params.relative_change_min = -0.001  # no step of this size passes
    xo = dom.conc0.copy()
    xo[0:2] = 5.0e4
    x = xo.copy()
    orc = O.Oracle(dom, dom.params.si())
    with capi.SedimentColumns.from_domain(dom) as g:
        g.set_state(x)
        g.run(200.0, 2, ADAPTIVE_EULER)
        f = g.ode_solver(g.get_state(), 200.0, ADAPTIVE_EULER)
        for _ in range(3):
            assert orc.ode_solver(xo, 200.0, ADAPTIVE_EULER) == 0
        assert orc.last_min_dt[0] <= dt_min
        assert np.all(np.isfinite(xo))
        assert np.array_equal(g.get_state(), xo)
        assert np.array_equal(f, orc.flux)
        assert g.last_min_dt() == orc.last_min_dt[0]
