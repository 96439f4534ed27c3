"""Fixed steps of launches on both sides of one wave per SIMD (65536 lanes), where
the kernels of some methods change to two; bitwise against the oracle."""
import numpy as np
import pytest

import oracle as O
from sedcol import capi, cases
from sedcol.params import EMP1, EMP2, EULER

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncol,K", [(4096, 7), (4097, 7), (2048, 17), (2050, 17), (1025, 33)])
@pytest.mark.parametrize("method,arith,weights,zw", [(EMP2, 0, 0, None), (EMP1, 1, 1, None),
                                                     (EMP1, 0, 0, capi.ZW_DEFAULTS), (EULER, 0, 0, capi.ZW_DEFAULTS)],
                         ids=["emp2-ref", "emp1-geo-fast", "emp1-ext", "euler-ext"])
def test_both_sides_of_a_full_device(gpu_ready, ncol, K, method, arith, weights, zw):
    dom = cases.plain_columns(ni=ncol, nj=1, K=K, seed=7)
    dom.params.arith, dom.params.emp_weights = arith, weights
    x = dom.conc0.copy()
    x[:5] += np.random.default_rng(ncol).uniform(10.0, 100.0, size=x[:5].shape)
    with capi.SedimentColumns.from_domain(dom) as g:
        if zw is not None:
            g.set_bioturbation_zw(zw)
        g.set_state(x)
        g.run(20.0, 3, method)
        xg, fg, bg = g.get_state(), g.fluxes(), g.budget()
    orc = O.Oracle(dom, dom.params.si(), zw=zw)
    assert orc.run(x, 20.0, 3, method, nthreads=4) == 0
    assert np.all(np.isfinite(x))
    assert np.array_equal(xg, x)
    assert np.array_equal(fg, orc.flux)
    assert np.array_equal(bg, orc.budget())
