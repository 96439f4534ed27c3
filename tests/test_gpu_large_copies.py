"""Copies through the shared pinned blocks: two handles at once, where one goes
the runtime's way, and large states of the transposed layout."""
import threading

import numpy as np
import pytest

from sedcol import capi, cases

pytestmark = pytest.mark.gpu


def test_two_handles_copy_at_once(gpu_ready):
    dom = cases.plain_columns(ni=400, nj=50, K=20, seed=1)  # 35 MB of state
    errors = []

    def work(seed):
        try:
            rng = np.random.default_rng(seed)
            with capi.SedimentColumns.from_domain(dom) as g:
                for _ in range(6):
                    x = rng.random(dom.conc0.shape)
                    g.set_state(x)
                    blob = g.save_checkpoint()
                    assert np.array_equal(g.get_state(), x)
                    g.set_state(dom.conc0)
                    g.load_checkpoint(blob)
                    assert np.array_equal(g.get_state(), x)
        except BaseException as e:  # reported by the test's own thread
            errors.append(e)

    team = [threading.Thread(target=work, args=(s,)) for s in (1, 2)]
    for t in team:
        t.start()
    for t in team:
        t.join()
    assert not errors, errors


@pytest.mark.parametrize("ncol,K", [(3251, 29), (3250, 30), (1490, 64), (95327, 1)])
def test_large_fortran_state_round_trip(gpu_ready, ncol, K):
    """States on both sides of 8 MiB and of whole blocks of 2 MiB."""
    x = np.random.default_rng(ncol).random((11, K, ncol))
    with capi.SedimentColumns(np.full(ncol, K, dtype=np.int32), np.zeros(ncol, dtype=np.int32), layout="fortran") as g:
        g.set_state(x)
        assert np.array_equal(g.get_state(), x)
