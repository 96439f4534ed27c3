"""The sweeps of the linearly implicit stepper leave their registers for the
general form when a value is not finite or a pivot is out of range.  A column
that does so must not change the column that shares its wave, nor may what an
earlier launch left in LDS enter the rows beyond a column; bitwise against the
oracle."""
import numpy as np
import pytest

import oracle as O
from sedcol import capi, spinup
from sedcol.params import ROS2_ADAPTIVE

pytestmark = pytest.mark.gpu


def _domain(layers, seed=17):
    rng = np.random.Generator(np.random.Philox(seed))
    dom = spinup.build(spinup.draw_inputs(rng, len(layers)), np.array(layers))
    dom.params.arith = 1
    dom.params.adaptive_method = ROS2_ADAPTIVE
    return dom


@pytest.mark.parametrize("block", [64, 256])
@pytest.mark.parametrize("layers,bad", [((24, 20), 0), ((24, 20), 1), ((17, 32), 0), ((32, 25, 18, 31, 17, 20), 3),
                                        ((40, 64, 33), 1)])
@pytest.mark.parametrize("span", [1.0, 30.0])
def test_column_beside_an_overflowing_one(gpu_ready, layers, bad, span, block):
    """Bottom water of 1e70 mmol/m3 oxygen: the rates of the first stage are
    finite, those of the second overflow."""
    dom = _domain(layers)
    dom.cbw[0, 5, bad] = 1.0e70
    sl = slice(dom.off[bad], dom.off[bad + 1])
    dom.conc0[5, sl] = 1.0e50
    with capi.SedimentColumns.from_domain(dom) as g:
        g.set_tuning([16, 32, 64], [block // 16, block // 32, block // 64])
        with pytest.raises(capi.SedcolError) as e:
            g.integrate(0.0, span)
        assert e.value.code == capi.SEDCOL_ENAN
        xg, dg = g.get_state(), g.diagnostics()
    orc = O.Oracle(dom, dom.params.si())
    xo = dom.conc0.copy()
    assert orc.emp_integrate(xo, span) == 1
    assert list(np.flatnonzero(orc.diag["status"])) == [bad]
    assert np.array_equal(dg["status"], orc.diag["status"])
    assert np.array_equal(xg, xo)
    for k in ("accepted", "rejected", "dt_next"):
        assert np.array_equal(dg[k], orc.diag[k]), k


def test_rows_beyond_a_column(gpu_ready):
    """Columns of 32 layers leave a factor that is not a number in row 23 of
    every place; the columns of 17 layers that follow there have pivots out of
    range, so they take their factor from LDS and their later solves run over 24
    rows."""
    n, m = 4096, 64
    dom = _domain(np.repeat([32, 17], [n, m]))
    dom.params.clamp = 0
    dom.params.D0 = 1.0e283
    dom.dzc[dom.off[:n] + 24] *= 1.0e-30
    with capi.SedimentColumns.from_domain(dom) as g:
        with pytest.raises(capi.SedcolError) as e:
            g.integrate(0.0, 1800.0)
        assert e.value.code == capi.SEDCOL_ENAN
        xg, dg = g.get_state(), g.diagnostics()
    sub = dom.subset(np.arange(n, n + m))
    orc = O.Oracle(sub, dom.params.si())
    xo = sub.conc0.copy()
    assert orc.emp_integrate(xo, 1800.0, nthreads=4) == 0
    assert np.all(np.isfinite(xo))
    assert np.all(dg["status"][:n] == 1) and np.all(dg["status"][n:] == 0)
    assert np.array_equal(xg[:, dom.off[n]:], xo)
    assert np.array_equal(dg["accepted"][n:], orc.diag["accepted"])
