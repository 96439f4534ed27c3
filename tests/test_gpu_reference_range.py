"""The reference form's right-hand side divides by reciprocals while every value
of a wave is in the range where that is exact, and by IEEE divisions otherwise:
both, and waves with columns of both kinds, bitwise against the oracle, at the
lane mappings' edges.  The adaptive Euler kernel at the sizes of its blocks."""
import numpy as np
import pytest

import oracle as O
from sedcol import capi, cases
from sedcol.params import ADAPTIVE_EULER, RUNGE_KUTTA_4

pytestmark = pytest.mark.gpu

LAYERS = np.array([1, 2, 16, 15, 3, 16, 17, 32, 31, 32, 33, 64, 63, 40])


def _state(kind, dom, rng):
    x = 10.0 ** rng.uniform(-3.0, 4.0, size=dom.conc0.shape)
    part = rng.random(x.shape) < 0.3
    if kind == "zeros":
        x[part] = 0.0
    elif kind == "negative":
        x[part] *= -1.0
    elif kind == "tiny":  # down to the denormals
        x[part] = 10.0 ** rng.uniform(-322.0, -100.0, size=int(part.sum()))
    elif kind == "edge":  # on both sides of the range's ends
        x[part] = 2.0 ** rng.choice([-501.0, -500.0, -499.0, -498.0, 490.0, 499.0, 500.0, 501.0], size=int(part.sum()))
    elif kind == "huge":
        x[part] = 10.0 ** rng.uniform(100.0, 300.0, size=int(part.sum()))
    elif kind == "one-column":  # a single layer outside in a single column
        x[:, dom.off[7] + 5] = 1.0e-200
    return x


def _domain(seed=3):
    rng = np.random.Generator(np.random.Philox(seed))
    dom = cases.build_columns(LAYERS, rng.uniform(0.1, 0.5, LAYERS.size), cases.draw_scalars(rng, LAYERS.size))
    dom.params.arith = 0
    return dom, rng


@pytest.mark.parametrize("kind", ["plain", "zeros", "negative", "tiny", "edge", "huge", "one-column", "rates",
                                  "closed"])
def test_rhs_ranges_bitwise(gpu_ready, kind):
    dom, rng = _domain()
    x = _state(kind, dom, rng)
    if kind == "rates":
        dom.params.kin.ksO2oxic = 1.0e-25
        dom.params.kin.kinNO3anox = 1.0e30
    if kind == "closed":
        dom.params.bcup_dis = dom.params.bcup_part = 3
        dom.params.bcdown = 2
    p = dom.params.si()
    with capi.SedimentColumns.from_domain(dom) as g:
        rg, fg = g.get_rhs(x)
    with np.errstate(all="ignore"):
        ro, fo = O.Oracle(dom, p).rhs(x)
    assert np.array_equal(rg, ro, equal_nan=True)
    assert np.array_equal(fg, fo, equal_nan=True)


def test_rk4_from_a_front_of_denormals_bitwise(gpu_ready):
    """From sediment without detritus the first steps carry values through the
    whole range down to the denormals, layer by layer."""
    dom, _ = _domain()
    dom.params.clamp = 1
    p = dom.params.si()
    xo = dom.conc0.copy()
    with capi.SedimentColumns.from_domain(dom) as g:
        g.run(60.0, 40, RUNGE_KUTTA_4)
        xg, bg = g.get_state(), g.budget()
    orc = O.Oracle(dom, p)
    assert orc.run(xo, 60.0, 40, RUNGE_KUTTA_4) == 0
    assert np.array_equal(xg, xo)
    assert np.array_equal(bg, orc.budget())


@pytest.mark.parametrize("ncol,K", [(1, 16), (4, 15), (5, 9), (2, 32), (3, 17), (8, 20), (9, 32), (16, 31), (1, 64),
                                    (2, 33), (8, 40)])
def test_adaptive_euler_block_sizes_bitwise(gpu_ready, ncol, K):
    dom = cases.plain_columns(ni=ncol, nj=1, K=K, seed=9)
    dom.params.dt_min = 1.0
    p = dom.params.si()
    xo = dom.conc0.copy()
    xo[0:2] = 5.0e4
    with capi.SedimentColumns.from_domain(dom) as g:
        g.set_state(xo)
        g.run(1800.0, 3, ADAPTIVE_EULER)
        xg, fg, bg, dg, lm = g.get_state(), g.fluxes(), g.budget(), g.diagnostics(), g.last_min_dt()
    orc = O.Oracle(dom, p)
    for _ in range(3):
        orc.ode_solver(xo, 1800.0, ADAPTIVE_EULER)
    assert np.array_equal(xg, xo)
    assert np.array_equal(fg, orc.flux)
    assert np.array_equal(bg, orc.budget())
    assert lm == orc.last_min_dt[0]
    for k in ("accepted", "dt_last", "dt_minacc"):
        assert np.array_equal(dg[k], orc.diag[k]), k
