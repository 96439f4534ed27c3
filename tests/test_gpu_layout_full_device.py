"""The transposed layout on a device without room for the array of the
transposition: the host transposes."""
import numpy as np
import pytest

from sedcol import ADAPTIVE_EULER, capi, cases

pytestmark = pytest.mark.gpu

NI, NJ, K = 100, 60, 32  # 17 MB of state


def _fill(leave):
    """Takes the free device memory but for about `leave` bytes."""
    import torch

    held = []
    for step in (1 << 30, 32 << 20, 2 << 20):
        room = (torch.cuda.mem_get_info()[0] - leave) // step * step
        if room > 0:
            held.append(torch.empty(room, dtype=torch.uint8, device="cuda"))
    return held


def test_state_and_rhs_on_a_full_device(gpu_ready):
    import torch

    dom = cases.plain_columns(ni=NI, nj=NJ, K=K, seed=4)
    x = dom.fortran_state(dom.conc0)
    with capi.SedimentColumns(dom.nlayers, dom.mask, layout="fortran") as g, \
            capi.SedimentColumns.from_domain(dom) as p, \
            capi.SedimentColumns(dom.nlayers, dom.mask, layout="fortran") as q:
        q.set_params(dom.params)
        q.set_geometry(*[a.reshape(dom.ncol, K).T for a in (dom.dz, dom.dzc, dom.phi, dom.phiI, dom.bfac)], dom.biot)
        q.set_forcing(*dom.record(0))
        q.set_state(x)
        q.run(1.0, 1, ADAPTIVE_EULER)  # allocates two of the three arrays of a right-hand side
        want, fwant = p.get_rhs(dom.conc0)
        torch.cuda.empty_cache()
        held = _fill(4 << 20)
        try:
            assert torch.cuda.mem_get_info()[0] < x.nbytes
            got_r, f = q.get_rhs(x)
            g.set_state(x)
            got = g.get_state()
        finally:
            held.clear()
            torch.cuda.empty_cache()
        assert np.array_equal(got, x)
        assert np.array_equal(got_r, dom.fortran_state(want)) and np.array_equal(f, fwant)
        # with room again the device transposes
        assert np.array_equal(g.get_state(), x)
