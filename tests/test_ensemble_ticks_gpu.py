"""The end of an ensemble's tick and the member totals, on MI355X: the tick is ended by the
last of the totals' workgroups, or by a launch of its own where a tick has none."""
import numpy as np
import pytest

from pihm_amd.ensemble import Ensemble
from pihm_amd.forcing import StormForcing, run_config
from pihm_amd.meshgen import make_watershed

pytestmark = pytest.mark.gpu


def _run(ms, fs, pieces):
    e = Ensemble(ms, fs, run_config(600.0))
    try:
        for k, m in enumerate(ms):
            e.set_state(k, m.initial_state())
        timed = [e.op_stats()["launches"]]
        for t in pieces:
            assert e.run(t) == 0
            timed.append(e.op_stats()["launches"])
        return [e.get_state(k) for k in range(len(ms))], timed, e.counters()["op_launches"]
    finally:
        e.close()


@pytest.mark.parametrize("nelem", [[40], [650, 700], [40, 650, 700, 1400, 5500]])
def test_ticks_of_any_membership(nelem):
    """Members of one chunk of 2,048 entries, of one chunk and a little, and of several, alone
    and together, in one run and in pieces: the same bits, and every run times launches."""
    ms = [make_watershed(n, seed=k + 1, n_seg=4) for k, n in enumerate(nelem)]
    fs = [StormForcing(4, seed=k, nelem=m.nelem, p_wet=0.7) for k, m in enumerate(ms)]
    print(f"[ens ticks] {nelem}", flush=True)
    whole, timed, launches = _run(ms, fs, [600.0])
    pieces, timed3, launches3 = _run(ms, fs, [120.0, 300.0, 600.0])
    assert 0 == timed[0] < timed[1] <= launches
    assert 0 == timed3[0] < timed3[1] < timed3[2] < timed3[3] <= launches3
    for k in range(len(ms)):
        assert np.array_equal(whole[k], pieces[k])
        alone, _, _ = _run(ms[k:k + 1], fs[k:k + 1], [600.0])
        assert np.array_equal(alone[0], whole[k])
