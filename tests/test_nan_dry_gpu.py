"""NaN derivatives of dry surfaces, on MI355X: a quotient of the overland flow that is not a
number is reported whether or not there is water on either side of the face."""
import copy

import numpy as np
import pytest

import oracle as O
from pihm_amd.mesh import DIFF_WAVE, KINEMATIC
from pihm_amd.meshgen import make_watershed
from pihm_amd.rhs import HipRHS

pytestmark = pytest.mark.gpu


def _mesh(kind, mode):
    base = make_watershed(535, seed=1, n_seg=20)
    m = copy.copy(base)
    m.a = {k: v.copy() for k, v in base.a.items()}
    m._keep = []
    m.surf_mode = mode
    inner = np.nonzero(np.all(m.a["nabr"] > 0, axis=1))[0]
    e = int(inner[len(inner) // 2])
    n = int(m.a["nabr"][e, 1]) - 1
    if kind == "rough":              # the mean over one face is zero
        m.a["rough"][[e, n]] = 0.0
    elif kind == "rough nan":
        m.a["rough"][e] = np.nan
    elif kind == "elevation":
        m.a["zmax"][e] = np.nan
    elif kind == "distance":         # a head difference over no distance, beside dry faces
        m.a["nabrdist"][e, 1] = 0.0
    elif kind == "edge":
        m.a["edge"][e, 1] = np.inf
    return m, e, n


@pytest.mark.parametrize("mode", [DIFF_WAVE, KINEMATIC])
@pytest.mark.parametrize("path", [0, 1])
@pytest.mark.parametrize("kind", ["sound", "rough", "rough nan", "elevation", "distance", "edge"])
def test_dry_faces_report_as_wet_ones(kind, path, mode):
    """Return code and the NaN components are the oracle's on a wholly dry surface, on one
    dry around the element, and on one that is wet there."""
    m, e, n = _mesh(kind, mode)
    ne = m.nelem
    near = {e, n} | {int(q) - 1 for k in (e, n) for q in m.a["nabr"][k] if q > 0}
    away = np.array([i not in near for i in range(ne)])
    for surf in (np.zeros(ne), np.where(away, 2e-2, 0.0), np.full(ne, 2e-2)):
        y = m.initial_state()
        y[:ne] = surf
        print(f"[nan dry] {kind} path {path} mode {mode} wet {int((surf > 0).sum())}", flush=True)
        h, o = HipRHS(m, rhs_path=path), O.OracleRHS(m)
        with np.errstate(all="ignore"):
            rc_h, dh = h.ode(y)
            rc_o, do = o.ode(y)[:2]
        h.close()
        assert rc_h == rc_o
        assert np.array_equal(np.isnan(dh), np.isnan(do))
        if kind == "sound":
            assert rc_h == 0 and not np.isnan(dh).any()
