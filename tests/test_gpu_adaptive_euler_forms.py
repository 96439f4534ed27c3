"""Adaptive Euler of domains that fill one workgroup of two waves per SIMD, in
every arithmetic form; bitwise against the oracle."""
import numpy as np
import pytest

import oracle as O
from sedcol import capi, cases
from sedcol.params import ADAPTIVE_EULER

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncol,K", [(17, 16), (32, 7), (9, 30), (5, 63)])
@pytest.mark.parametrize("arith,zw", [(0, None), (1, None), (0, capi.ZW_DEFAULTS)], ids=["ref", "fast", "ext"])
def test_forms_bitwise(gpu_ready, ncol, K, arith, zw):
    dom = cases.plain_columns(ni=ncol, nj=1, K=K, seed=9)
    dom.params.dt_min = 1.0
    dom.params.arith = arith
    xo = dom.conc0.copy()
    xo[:5] += 50.0
    with capi.SedimentColumns.from_domain(dom) as g:
        if zw is not None:
            g.set_bioturbation_zw(zw)
        g.set_state(xo)
        g.run(1800.0, 3, ADAPTIVE_EULER)
        xg, fg, bg, lm = g.get_state(), g.fluxes(), g.budget(), g.last_min_dt()
    orc = O.Oracle(dom, dom.params.si(), zw=zw)
    for _ in range(3):
        orc.ode_solver(xo, 1800.0, ADAPTIVE_EULER)
    assert np.all(np.isfinite(xo))
    assert np.array_equal(xg, xo)
    assert np.array_equal(fg, orc.flux)
    assert np.array_equal(bg, orc.budget())
    assert lm == orc.last_min_dt[0]
