"""The NaN report after an unrelated HIP call of the same thread has failed, on MI355X."""
import ctypes as C

import pytest

from pihm_amd.meshgen import make_watershed
from pihm_amd.rhs import HipRHS
from test_nan_report_gpu import _adverse_outlet

pytestmark = pytest.mark.gpu


def test_an_earlier_error_is_not_the_reports():
    """A failed call elsewhere (a device number that does not exist, refused by the runtime on
    the host) leaves its error with the thread; polls then and later still belong to their
    own evaluations."""
    m, bad = make_watershed(40, seed=1, n_seg=4), _adverse_outlet(40, 4)
    a, b = HipRHS(m), HipRHS(bad)
    hip = C.CDLL(None)     # the runtime that the library has loaded
    ya, yb = m.initial_state(), bad.initial_state()
    try:
        assert a.ode(ya)[0] == 0 and b.ode(yb)[0] == 1
        for h in (a, b):
            print("[nan poll]", flush=True)
            assert hip.hipSetDevice(9999) != 0
            assert h.L.pihm_ctx_poll_nan(h.ctx) == 0
            hip.hipGetLastError()
        for _ in range(3):
            assert a.ode(ya)[0] == 0 and b.ode(yb)[0] == 1
            assert a.L.pihm_ctx_poll_nan(a.ctx) == 0 and b.L.pihm_ctx_poll_nan(b.ctx) == 0
    finally:
        a.close()
        b.close()
