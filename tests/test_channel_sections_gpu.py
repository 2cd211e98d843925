"""Channel sections of one shape each, from dry to deep and narrow to wide, on MI355X against
the oracle: the powers of the sections that are not rectangles are worked in step."""
import copy

import numpy as np
import pytest

import oracle as O
from conftest import assert_rhs_close
from pihm_amd.mesh import CUBIC, QUADRATIC, RECTANGLE, TRIANGLE
from pihm_amd.rhs import HipRHS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path", [0, 1])
@pytest.mark.parametrize("coeff", [1e-3, 0.3, 40.0, 0.0, -0.5, np.nan])
@pytest.mark.parametrize("shape", [RECTANGLE, TRIANGLE, QUADRATIC, CUBIC])
def test_sections_of_one_shape(c0, shape, coeff, path):
    """1e-12 of the assembled terms, as every RHS value; NaN, where a coefficient makes no
    section, in the oracle's components."""
    m = copy.copy(c0)
    m.a = dict(c0.a)
    m._keep = []
    ne, nr = m.nelem, m.nriver
    rng = np.random.default_rng(shape)
    m.a["intrpl_ord"] = np.full(nr, shape, np.int32)
    m.a["coeff"] = coeff * rng.uniform(0.5, 2.0, nr)
    y = m.initial_state()
    y[:ne] = rng.uniform(0.0, 2e-2, ne)
    y[3 * ne:3 * ne + nr] = np.where(rng.random(nr) < 0.2, 0.0, 10 ** rng.uniform(-6, 1.5, nr))
    print(f"[sections] shape {shape} coeff {coeff} path {path}", flush=True)
    h, o = HipRHS(m, rhs_path=path), O.OracleRHS(m)
    rc_h, dh = h.ode(y)
    with np.errstate(all="ignore"):
        rc_o, do, mag = o.ode(y, with_mag=True)
    h.close()
    assert rc_h == rc_o
    fin = np.isfinite(do) & np.isfinite(mag)
    assert np.array_equal(np.isnan(dh[~fin]), np.isnan(do[~fin]))
    assert_rhs_close(dh[fin], do[fin], mag[fin], 1e-12, f"shape {shape} coeff {coeff}")
