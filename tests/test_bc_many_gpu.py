"""Boundary conditions on either side of the line where the series are interpolated in a
launch of their own, on MI355X, bit for bit against the oracle."""
import numpy as np
import pytest

import oracle as O
from pihm_amd.bc import HipBC
from pihm_amd.rhs import HipRHS
from test_bc_gpu import T0, _series

pytestmark = pytest.mark.gpu
DIRECT = 16384     # entries with a series up to which each interpolates its own


@pytest.mark.parametrize("sets", ["both", "edges", "rivers of few"])
@pytest.mark.parametrize("coded", [DIRECT - 1, DIRECT, DIRECT + 1, None])
def test_many_entries_with_a_series(tree_small, coded, sets):
    m = tree_small
    ne, nr = m.nelem, m.nriver
    rng = np.random.default_rng(coded or 1)
    code = (rng.choice([-1, 1], 3 * ne) * rng.integers(1, 300, 3 * ne)).astype(np.int32)
    rcode = np.zeros(nr, np.int32)
    if sets == "both":
        rcode = (rng.choice([-1, 1], nr) * rng.integers(1, 4, nr)).astype(np.int32)
    elif sets == "rivers of few":
        rcode[::7] = 2
    if coded:
        off = rng.permutation(3 * ne)[:3 * ne + int((rcode != 0).sum()) - coded]
        code[off] = 0
        assert int((code != 0).sum() + (rcode != 0).sum()) == coded
    code = code.reshape(ne, 3)
    ets = _series(299, 40, rng.uniform(100, 200, 299), 3.0, 4)
    rts = None if sets == "edges" else _series(3, 2, [1.0, 2.0, 3.0], 0.5, 5, dt=7200.0)
    print(f"[bc many] {coded} {sets}", flush=True)
    h = HipRHS(m)
    eb, rb = rng.normal(size=(ne, 3)), rng.normal(size=nr)
    h.set_step_inputs(elem_bc=eb.ravel(), river_bc=rb)
    b = HipBC(h, code, ets, rcode, rts)
    try:
        end = min(s[0][:, -1].min() for s in (ets, rts) if s is not None)
        for t in (T0, T0 + 0.37 * (end - T0), end):
            assert b.apply(t) == 0
            ge, gr = b.values()
            rc, eb, rb = O.bc_apply(ne, nr, t, code, ets, rcode, rts, eb, rb)
            assert rc == 0
            assert np.array_equal(ge, eb) and np.array_equal(gr, rb)
        # neither a time past the series nor one that is no number changes an entry
        assert b.apply(end + 1.0) != 0
        assert b.apply(float("nan")) == 0
        ge, gr = b.values()
        assert np.array_equal(ge, eb) and np.array_equal(gr, rb)
    finally:
        b.close()
        h.close()
