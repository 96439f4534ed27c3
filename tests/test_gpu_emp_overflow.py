"""An adaptive step whose two estimates are both infinite is an error in every
kernel shape, as in the oracle, and leaves the state as it was: a single layer
with a prescribed influx of phosphate and, so that the rate of the infinite
estimate is not negative, a negative adsorption rate."""
import numpy as np
import pytest

import oracle as O
from sedcol import capi, cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layers_per_lane", [1, 2])
@pytest.mark.parametrize("arith", [0, 1])
@pytest.mark.parametrize("layers", [(1, 1, 1), (1, 8, 1)])
def test_infinite_estimates(gpu_ready, layers, arith, layers_per_lane):
    rng = np.random.Generator(np.random.Philox(1))
    dom = cases.build_columns(np.array(layers), np.full(3, 0.1), cases.draw_scalars(rng, 3))
    dom.params.arith = arith
    dom.params.bcup_dis = 1
    dom.params.kin.PAds = -0.01
    dom.fup[0, 5:10] = 0.0
    dom.fup[0, 9, 2] = 1.0e305 * dom.dz[-1] * dom.phi[-1]
    dom.conc0[5] = 200.0
    dom.conc0[9] = 1.0
    with capi.SedimentColumns.from_domain(dom) as g:
        g.set_tuning([16, 32, 64], [16, 8, 4], [layers_per_lane] * 3)
        with pytest.raises(capi.SedcolError) as e:
            g.integrate(0.0, 3600.0)
        assert e.value.code == capi.SEDCOL_ENAN
        xg, dg = g.get_state(), g.diagnostics()
    orc = O.Oracle(dom, dom.params.si())
    xo = dom.conc0.copy()
    assert orc.emp_integrate(xo, 3600.0) == 1
    assert list(orc.diag["status"]) == [0, 0, 1] and np.all(np.isfinite(xo))
    assert np.array_equal(dg["status"], orc.diag["status"])
    assert np.array_equal(dg["accepted"], orc.diag["accepted"])
    assert np.array_equal(xg, xo)
