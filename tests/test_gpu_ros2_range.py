"""The transport factor of the linearly implicit stepper outside the range of
its fast reciprocals: with a molecular diffusivity near the largest double the
pivots of the dissolved species leave that range and the wave repeats the
solve with divisions.  Columns whose wave mixes layer counts, and the lane
mappings' edges; bitwise against the oracle."""
import numpy as np
import pytest

import oracle as O
from sedcol import capi, spinup
from sedcol.params import ROS2_ADAPTIVE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d0", [0.9, 1.0e283])
@pytest.mark.parametrize("layers", [(17, 32, 24, 25), (33, 64, 40, 41), (16, 8, 1, 3)], ids=["lpc32", "lpc64", "lpc16"])
def test_ros2_pivot_range_bitwise(gpu_ready, layers, d0):
    rng = np.random.Generator(np.random.Philox(17))
    s = spinup.draw_inputs(rng, len(layers))
    dom = spinup.build(s, np.array(layers))
    dom.params.arith = 1
    dom.params.clamp = 0
    dom.params.D0 = d0
    dom.params.adaptive_method = ROS2_ADAPTIVE
    p = dom.params.si()
    with capi.SedimentColumns.from_domain(dom) as g:
        g.integrate(0.0, 1800.0)
        xg, dg = g.get_state(), g.diagnostics()
    orc = O.Oracle(dom, p)
    xo = dom.conc0.copy()
    assert orc.emp_integrate(xo, 1800.0, nthreads=4) == 0
    assert np.all(np.isfinite(xo))
    assert np.array_equal(xg, xo)
    assert np.array_equal(dg["accepted"], orc.diag["accepted"])
    assert np.array_equal(dg["rejected"], orc.diag["rejected"])
