"""sedcol_step of small domains goes through pinned staging, larger ones through
copies: the same results on both sides of the limit, in both layouts, for every
fixed-step method, with the land, error and aliasing cases of the call."""
import numpy as np
import pytest

import oracle as O
from sedcol import capi, cases

pytestmark = pytest.mark.gpu

# 512 KiB of staging hold 5957 cells and columns of 11 values
SHAPES = [(1, 1, 15), (4, 4, 30), (3, 5, 64), (73, 5, 15), (73, 5, 16), (40, 20, 9)]


def _fortran(dom, K):
    g = capi.SedimentColumns(dom.nlayers, dom.mask, layout="fortran")
    g.set_params(dom.params)
    g.set_geometry(*[a.reshape(dom.ncol, K).T for a in (dom.dz, dom.dzc, dom.phi, dom.phiI, dom.bfac)], dom.biot)
    g.set_forcing(*dom.record(0))
    return g


@pytest.mark.parametrize("layout", ["packed", "fortran"])
@pytest.mark.parametrize("ni,nj,K", SHAPES)
def test_step_bitwise(gpu_ready, ni, nj, K, layout):
    dom = cases.plain_columns(ni=ni, nj=nj, K=K, seed=2)
    if dom.ncol > 2:
        dom.mask[1] = 1
    p = dom.params.si()
    wet = np.repeat(dom.mask, dom.nlayers) == 0
    g = capi.SedimentColumns.from_domain(dom) if layout == "packed" else _fortran(dom, K)
    with g:
        for method in (0, 1, 2, 3, 4, 5):
            xo = dom.conc0.copy()
            orc = O.Oracle(dom, p)
            x = xo.copy() if layout == "packed" else dom.fortran_state(xo).copy()
            g.reset_diagnostics()
            for _ in range(2):
                f = g.ode_solver(x, 60.0, method)
                assert orc.ode_solver(xo, 60.0, method) == 0
            xg = x if layout == "packed" else dom.packed_state(x)
            assert np.array_equal(xg[:, wet], xo[:, wet]), method
            assert np.array_equal(xg[:, ~wet], dom.conc0[:, ~wet]), method
            assert np.array_equal(f[:, dom.mask == 0], orc.flux[:, dom.mask == 0]), method
            if method == 2:
                assert g.last_min_dt() == orc.last_min_dt[0]
            assert np.array_equal(g.get_state(), x), method


def test_step_errors_leave_the_state(gpu_ready):
    dom = cases.plain_columns(ni=2, nj=2, K=12, seed=3)
    with capi.SedimentColumns.from_domain(dom) as g:
        for dt in (0.0, -1.0, np.inf, np.nan):
            x = dom.conc0.copy()
            with pytest.raises(capi.SedcolError) as e:
                g.ode_solver(x, dt, 1)
            assert e.value.code == capi.SEDCOL_EINVAL and np.array_equal(x, dom.conc0)
        x = dom.conc0.copy()
        x[5, 3] = np.nan
        with pytest.raises(capi.SedcolError) as e:
            g.ode_solver(x, 60.0, 1)
        assert e.value.code == capi.SEDCOL_ENAN


def test_rhs_over_its_own_input(gpu_ready):
    """The output may be, or overlap, the input."""
    dom = cases.plain_columns(ni=330, nj=100, K=20, seed=4)  # 58 MB: through the pinned blocks
    want, _ = O.Oracle(dom, dom.params.si()).rhs(dom.conc0)
    with capi.SedimentColumns.from_domain(dom) as g:
        for shift in (0, 5, dom.conc0.size):
            buf = np.empty(dom.conc0.size + shift)
            src, dst = buf[:dom.conc0.size], buf[shift:]
            src[...] = dom.conc0.ravel()
            f = np.empty((11, dom.ncol)) if shift != dom.conc0.size else None
            if shift == dom.conc0.size:  # apart
                dst = np.empty(dom.conc0.size)
            capi.check(capi.lib().sedcol_rhs(g._h, capi._pd(src), capi._pd(dst), capi._pd(f) if f is not None else None))
            assert np.array_equal(dst, want.ravel()), shift


@pytest.mark.parametrize("ncol,K", [(1, 1), (63, 64), (64, 1), (65, 17), (200, 33)])
def test_fortran_state_round_trip(gpu_ready, ncol, K):
    dom = cases.plain_columns(ni=ncol, nj=1, K=K, seed=5)
    x = np.random.default_rng(0).random((11, K, ncol))
    with _fortran(dom, K) as g:
        g.set_state(x)
        assert np.array_equal(g.get_state(), x)
        rg, fg = g.get_rhs(x)
    ro, fo = O.Oracle(dom, dom.params.si()).rhs(dom.packed_state(x))
    assert np.array_equal(dom.packed_state(rg), ro) and np.array_equal(fg, fo)
