"""The kernel shape of an untuned handle is the one that sedcol_get_tuning reports,
for each adaptive method, so installing it again changes nothing."""
import numpy as np
import pytest

from sedcol import capi, cases
from sedcol.params import EMP_ADAPTIVE, ROS2_ADAPTIVE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method,threads", [(EMP_ADAPTIVE, 256), (ROS2_ADAPTIVE, 64)])
def test_default_shape_is_reported(gpu_ready, method, threads):
    dom = cases.ragged_columns(40, seed=3)
    dom.params.adaptive_method = method
    with capi.SedimentColumns.from_domain(dom) as g:
        t = g.get_tuning()
        assert [a * b for a, b in zip(t["lanes_per_column"], t["columns_per_group"])] == [threads] * 3
        g.integrate(0.0, 600.0)
        x = g.get_state()
        g.set_tuning(t["lanes_per_column"], t["columns_per_group"], t["layers_per_lane"])
        assert g.get_tuning() == t
        g.set_state(dom.conc0)
        g.reset_diagnostics()
        g.integrate(0.0, 600.0)
        assert np.array_equal(g.get_state(), x)


def test_installed_shape_holds_for_both_methods(gpu_ready):
    dom = cases.ragged_columns(40, seed=3)
    with capi.SedimentColumns.from_domain(dom) as g:
        g.set_tuning([16, 32, 64], [8, 4, 2])
        want = g.get_tuning()
        dom.params.adaptive_method = ROS2_ADAPTIVE
        g.set_params(dom.params)
        assert g.get_tuning() == want
