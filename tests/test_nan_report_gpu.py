"""The NaN flag's report to the host, call after call and context after context, on MI355X."""
import numpy as np
import pytest

from pihm_amd.meshgen import make_watershed
from pihm_amd.rhs import HipRHS

pytestmark = pytest.mark.gpu


def _adverse_outlet(n, seg):
    """A zero-depth-gradient outlet on an adverse bed slope: the derivative of a full
    river is NaN there, that of a dry one is not."""
    m = make_watershed(n, seed=1, n_seg=seg)
    to = m.rivers["tonode"][int(np.nonzero(m.rivers["down"] < 0)[0][0])] - 1
    m.node_zmax[to] += 3.0
    m.node_zmin[to] += 3.0
    m.a = None
    m.init()
    return m


@pytest.mark.parametrize("n,seg", [(40, 4), (535, 20)])
def test_report_belongs_to_its_call(n, seg):
    """Every call reports its own derivative's NaN and no other's: two contexts in turn, one
    whose derivative is NaN and one whose is not, and on each the first, second and later
    calls; a poll without an evaluation in between finds the flag cleared."""
    print(f"[nan report] n {n}", flush=True)
    bad, good = _adverse_outlet(n, seg), make_watershed(n, seed=1, n_seg=seg)
    a, b = HipRHS(bad), HipRHS(good)
    try:
        ya, yb = bad.initial_state(), good.initial_state()
        for _ in range(4):
            assert a.ode(ya)[0] == 1
            assert a.L.pihm_ctx_poll_nan(a.ctx) == 0
            assert b.ode(yb)[0] == 0
            assert b.L.pihm_ctx_poll_nan(b.ctx) == 0
    finally:
        a.close()
        b.close()
