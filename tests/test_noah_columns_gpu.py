"""The Noah kernels' workgroups of 64 columns at the ends of their range, on MI355X: meshes
whose last workgroup holds one column, a few, or all but one, against the oracle."""
import numpy as np
import pytest

import test_noahlsm_gpu as lsm
import test_noahsoil_gpu as soil
from pihm_amd.meshgen import make_watershed

pytestmark = pytest.mark.gpu


class _Mesh:
    def __init__(self, m):
        self.m = m

    def getfixturevalue(self, _):
        return self.m


@pytest.mark.parametrize("n", [20, 63, 64, 65, 130])
def test_columns_of_partial_workgroups(n):
    """Both steps at their usual tolerances; every layer count from 2 to 11 is drawn."""
    m = make_watershed(n, seed=2, n_seg=3)
    name = f"n={n} ({m.nelem} columns)"
    soil.test_noah_soil_step_parity(name, _Mesh(m))
    lsm.test_noah_step_parity_chained(name, 1.0, _Mesh(m))
