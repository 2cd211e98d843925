"""Mesh descriptors whose fields share one array, on MI355X: a caller may pass the same
array for several fields, and each field keeps its own values."""
import copy

import numpy as np
import pytest

from pihm_amd.meshgen import make_watershed
from pihm_amd.rhs import HipRHS

pytestmark = pytest.mark.gpu


def _mesh(base, **fields):
    """A copy of a mesh with some fields replaced, not copied: desc() passes their own
    pointers on."""
    m = copy.copy(base)
    m.a = dict(base.a)
    m.a.update(fields)
    m._keep = []
    return m


def _ode(m, y, path):
    h = HipRHS(m, rhs_path=path, record=True)
    rng = np.random.default_rng(2)
    u = lambda top: rng.uniform(0.0, top, m.nelem)
    h.set_step_inputs(pcpdrp=u(3e-6), ws0_surf=u(1e-2), edir=u(1e-8), ett=u(1e-8))
    rc, dy = h.ode(y)
    h.close()
    assert rc == 0
    return dy


@pytest.mark.parametrize("path", [0, 1])
@pytest.mark.parametrize("names", [("kmach", "kmacv"), ("kmach", "dmac"), ("kmach", "ksath", "ksatv", "kmacv"),
                                   ("areafv", "areafh"), ("kmach", "rough", "rzd")])
def test_fields_of_one_array(names, path):
    """The derivative with the fields in one array equals, bit for bit, the one with the
    same values in arrays of their own.  The water table lies anywhere from a third of the soil
    to above it, in the macropores and the root zone or not, so that every one of the fields
    is read."""
    base = make_watershed(535, seed=1, n_seg=20)
    ne = base.nelem
    # no macropores (zeros), or one positive value for what must not be zero
    v = np.zeros(ne) if "dmac" in names else np.random.default_rng(1).uniform(0.05, 0.2, ne)
    one = _mesh(base, **{k: v for k in names})
    own = _mesh(base, **{k: v.copy() for k in names})
    d = one.desc()
    p = {k: np.ctypeslib.as_array(getattr(d, k), (1,)).ctypes.data for k in names}
    assert len(set(p.values())) == 1
    y = base.initial_state()
    rng = np.random.default_rng(0)
    y[:ne] = rng.uniform(0.0, 2e-2, ne)
    y[2 * ne:3 * ne] = base.a["depth"] * rng.uniform(0.3, 1.1, ne)
    y[ne:2 * ne] = 0.7 * np.maximum(base.a["depth"] - y[2 * ne:3 * ne], 0.0)
    print(f"[shared fields] {names} path {path}", flush=True)
    assert np.array_equal(_ode(one, y, path), _ode(own, y, path))
